// Queries and keys normed over their whole projection, rotated in neighbouring pairs, and the cache write, in one pass.
//
// Per token, from the float32 result of the fused q, k projection [T, (nh + nkv) hd]:
//   q <- q / sqrt(mean(q^2 over all nh hd columns) + eps) * wq,   k likewise over its nkv hd columns with wk;
//   columns (2i, 2i + 1), i < rot_dim / 2, of every head become (u cos a - v sin a, v cos a + u sin a) with
//   a = position * inv_freq[i]  (angles, sines and cosines in float32; the other columns pass unchanged);
//   q goes to q_out [T, nh hd] in the activation dtype, the rotated k into the key tiles, and the values' tiles
//   receive either the k projection as it left the product (values tied to the keys) or nothing.
// The heads may leave wider than they came (hd_out >= hd): the columns beyond hd are zeros in q_out and in both
// tiles, so that head sizes which the attention kernels do not take run as the next size they do take (zeros add
// nothing to a score, and a value's zero columns meet zero columns of the output projection).
// The tiles' element order is the attention kernels' (cache_layout.h).  One workgroup a token.
#include "common.h"
#include "cache_layout.h"

using namespace atoma;

template <typename TQ, typename TC>
__global__ void __launch_bounds__(256)
qk_norm_rope_kernel(const float* __restrict__ qk, int ld, const int32_t* __restrict__ positions,
                    const float* __restrict__ inv_freq, int rot_dim, const float* __restrict__ wq,
                    const float* __restrict__ wk, float eps, TQ* __restrict__ q_out, int ldq, TC* __restrict__ kcache,
                    TC* __restrict__ vcache, const int32_t* __restrict__ slot_mapping, int page_size, int nh, int nkv,
                    int hd, int hd_out) {
  __shared__ float scratch[4];
  __shared__ float cs[128], sn[128];
  const int t = blockIdx.x;
  const float* row = qk + (size_t)t * ld;
  const int nq = nh * hd, nk = nkv * hd;
  float sq = 0.f, sk = 0.f;
  for (int i = threadIdx.x; i < nq; i += 256) sq += row[i] * row[i];
  for (int i = threadIdx.x; i < nk; i += 256) sk += row[nq + i] * row[nq + i];
  sq = block_sum<4>(sq, scratch);
  sk = block_sum<4>(sk, scratch);
  const float iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
  const float p = (float)positions[t];
  for (int i = threadIdx.x; i < rot_dim / 2; i += 256) {
    float s, c;
    sincosf(p * inv_freq[i], &s, &c);
    cs[i] = c, sn[i] = s;
  }
  __syncthreads();
  // a thread takes a pair of neighbouring columns
  for (int pr = threadIdx.x; pr < nq / 2; pr += 256) {
    const int col = 2 * pr, head = col / hd, d = col % hd;
    float u = row[col] * iq * wq[col], v = row[col + 1] * iq * wq[col + 1];
    if (d < rot_dim) {
      const float c = cs[d >> 1], s = sn[d >> 1];
      const float u2 = u * c - v * s;
      v = v * c + u * s;
      u = u2;
    }
    q_out[(size_t)t * ldq + head * hd_out + d] = from_f32<TQ>(u);
    q_out[(size_t)t * ldq + head * hd_out + d + 1] = from_f32<TQ>(v);
  }
  const int pad = hd_out - hd;
  for (int i = threadIdx.x; i < nh * pad; i += 256)
    q_out[(size_t)t * ldq + (i / pad) * hd_out + hd + i % pad] = from_f32<TQ>(0.f);
  if (kcache == nullptr) return;
  const int slot = slot_mapping[t];
  const int page = slot / page_size, off = slot % page_size;
  for (int pr = threadIdx.x; pr < nk / 2; pr += 256) {
    const int col = 2 * pr, head = col / hd, d = col % hd;
    const float r0 = row[nq + col], r1 = row[nq + col + 1];
    float u = r0 * ik * wk[col], v = r1 * ik * wk[col + 1];
    if (d < rot_dim) {
      const float c = cs[d >> 1], s = sn[d >> 1];
      const float u2 = u * c - v * s;
      v = v * c + u * s;
      u = u2;
    }
    const size_t tile = ((size_t)page * nkv + head) * page_size * hd_out;
    TC* kt = kcache + tile;
    kt[key_offset(off, d, page_size)] = from_f32<TC>(u);
    kt[key_offset(off, d + 1, page_size)] = from_f32<TC>(v);
    if (vcache != nullptr) {
      TC* vt = vcache + tile;
      vt[value_offset(d, off, hd_out, page_size)] = from_f32<TC>(r0);
      vt[value_offset(d + 1, off, hd_out, page_size)] = from_f32<TC>(r1);
    }
  }
  for (int i = threadIdx.x; i < nkv * pad; i += 256) {
    const int head = i / pad, d = hd + i % pad;
    const size_t tile = ((size_t)page * nkv + head) * page_size * hd_out;
    kcache[tile + key_offset(off, d, page_size)] = from_f32<TC>(0.f);
    if (vcache != nullptr) vcache[tile + value_offset(d, off, hd_out, page_size)] = from_f32<TC>(0.f);
  }
}

// The same where a row's pairs of columns are at most P a thread and two neighbours can be fetched and stored together (even sizes and
// strides): a thread keeps its pairs in registers, and row, weights, position and slot are one trip to memory.  Eight tokens of 32 + 8
// heads of 64: 7.4 us, 8.7 with the row read twice and the weights behind the sums; 2,048 tokens 15.0 and 18.8.
template <typename T> __device__ __forceinline__ void put2(T* p, float a, float b) {
  if constexpr (sizeof(T) == 2) {
    *reinterpret_cast<uint32_t*>(p) = f32_to_bf16_bits(a) | (uint32_t)f32_to_bf16_bits(b) << 16;
  } else {
    *reinterpret_cast<float2*>(p) = make_float2(a, b);
  }
}

template <int P, typename TQ, typename TC>
__global__ void __launch_bounds__(256)
qk_norm_rope_pairs_kernel(const float* __restrict__ qk, int ld, const int32_t* __restrict__ positions,
                          const float* __restrict__ inv_freq, int rot_dim, const float* __restrict__ wq,
                          const float* __restrict__ wk, float eps, TQ* __restrict__ q_out, int ldq, TC* __restrict__ kcache,
                          TC* __restrict__ vcache, const int32_t* __restrict__ slot_mapping, int page_size, int nh, int nkv,
                          int hd, int hd_out) {
  __shared__ float sums[2][4];
  __shared__ float cs[128], sn[128];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* row = qk + (size_t)t * ld;
  const int nq = nh * hd, nk = nkv * hd, pairs = (nq + nk) / 2;
  const int pos = positions[t], slot = kcache != nullptr ? slot_mapping[t] : 0;
  float2 x[P], w[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int c = 2 * min(tid + j * 256, pairs - 1);
    x[j] = *reinterpret_cast<const float2*>(row + c);
    w[j] = *reinterpret_cast<const float2*>(c < nq ? wq + c : wk + c - nq);
  }
  for (int i = tid; i < rot_dim / 2; i += 256) {
    float s, c;
    sincosf((float)pos * inv_freq[i], &s, &c);
    cs[i] = c, sn[i] = s;
  }
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int c = 2 * (tid + j * 256);
    const float both = fmaf(x[j].x, x[j].x, x[j].y * x[j].y);
    sq += c < nq ? both : 0.f;
    sk += c >= nq && c < nq + nk ? both : 0.f;
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) sums[0][wave] = sq, sums[1][wave] = sk;
  lds_barrier();
  sq = sk = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) sq += sums[0][i], sk += sums[1][i];
  const float iq = 1.0f / sqrtf(sq / (float)nq + eps), ik = 1.0f / sqrtf(sk / (float)nk + eps);
  const int page = slot / page_size, off = slot % page_size;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int c = 2 * (tid + j * 256);
    if (c >= nq + nk || (c >= nq && kcache == nullptr)) continue;
    const bool is_q = c < nq;
    const int col = is_q ? c : c - nq, head = col / hd, d = col % hd;
    const float inv = is_q ? iq : ik;
    float u = x[j].x * inv * w[j].x, v = x[j].y * inv * w[j].y;
    if (d < rot_dim) {
      const float cc = cs[d >> 1], s = sn[d >> 1];
      const float u2 = u * cc - v * s;
      v = v * cc + u * s;
      u = u2;
    }
    if (is_q) {
      put2(q_out + (size_t)t * ldq + head * hd_out + d, u, v);
    } else {
      const size_t tile = ((size_t)page * nkv + head) * page_size * hd_out;
      put2(kcache + tile + key_offset(off, d, page_size), u, v);
      if (vcache != nullptr) {
        vcache[tile + value_offset(d, off, hd_out, page_size)] = from_f32<TC>(x[j].x);
        vcache[tile + value_offset(d + 1, off, hd_out, page_size)] = from_f32<TC>(x[j].y);
      }
    }
  }
  const int pad = hd_out - hd;
  if (pad == 0) return;
  for (int i = tid; i < nh * pad; i += 256) q_out[(size_t)t * ldq + (i / pad) * hd_out + hd + i % pad] = from_f32<TQ>(0.f);
  if (kcache == nullptr) return;
  for (int i = tid; i < nkv * pad; i += 256) {
    const int head = i / pad, d = hd + i % pad;
    const size_t tile = ((size_t)page * nkv + head) * page_size * hd_out;
    kcache[tile + key_offset(off, d, page_size)] = from_f32<TC>(0.f);
    if (vcache != nullptr) vcache[tile + value_offset(d, off, hd_out, page_size)] = from_f32<TC>(0.f);
  }
}

extern "C" int atoma_qk_norm_rope(const float* qk, int ld, const int32_t* positions, const float* inv_freq, int rot_dim,
                                  const float* wq, const float* wk, float eps, void* q_out, int ldq, int q_dtype,
                                  void* kcache, void* vcache, int cache_dtype, const int32_t* slot_mapping,
                                  int page_size, int n_tokens, int nh, int nkv, int hd, int hd_out,
                                  hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (hd <= 0 || hd % 2 || rot_dim < 0 || rot_dim % 2 || rot_dim > hd || rot_dim > 256 || nh <= 0 || nkv <= 0 ||
      page_size <= 0 || ld < (nh + nkv) * hd || hd_out < hd || ldq < nh * hd_out)
    return ATOMA_ERR_SHAPE;
  dim3 grid(n_tokens), block(256);
  const int pairs = (nh + nkv) * hd / 2, per = (pairs + 255) / 256;
  // (the weights' and the row's pairs are eight bytes, those of the outputs two elements; an element of the cache is as wide as one of q)
  const bool in_pairs = per <= 8 && ld % 2 == 0 && ldq % 2 == 0 && hd_out % 2 == 0 &&
                        (((uintptr_t)qk | (uintptr_t)wq | (uintptr_t)wk | (uintptr_t)q_out | (uintptr_t)kcache) & 7) == 0;
#define ATOMA_QKN_PAIRS(P, TQ, TC)                                                                                          \
  hipLaunchKernelGGL((qk_norm_rope_pairs_kernel<P, TQ, TC>), grid, block, 0, stream, qk, ld, positions, inv_freq, rot_dim, \
                     wq, wk, eps, (TQ*)q_out, ldq, (TC*)kcache, (TC*)vcache, slot_mapping, page_size, nh, nkv, hd, hd_out)
  if (in_pairs && q_dtype == cache_dtype && (q_dtype == kF32 || q_dtype == kBF16)) {
    if (q_dtype == kF32) {
      if (per <= 3) ATOMA_QKN_PAIRS(3, float, float);
      else if (per <= 5) ATOMA_QKN_PAIRS(5, float, float);
      else ATOMA_QKN_PAIRS(8, float, float);
    } else {
      if (per <= 3) ATOMA_QKN_PAIRS(3, bf16_t, bf16_t);
      else if (per <= 5) ATOMA_QKN_PAIRS(5, bf16_t, bf16_t);
      else ATOMA_QKN_PAIRS(8, bf16_t, bf16_t);
    }
    ATOMA_LAUNCH_CHECK();
    return 0;
  }
#undef ATOMA_QKN_PAIRS
#define ATOMA_QKN(TQ, TC)                                                                                          \
  hipLaunchKernelGGL((qk_norm_rope_kernel<TQ, TC>), grid, block, 0, stream, qk, ld, positions, inv_freq, rot_dim, \
                     wq, wk, eps, (TQ*)q_out, ldq, (TC*)kcache, (TC*)vcache, slot_mapping, page_size, nh, nkv, hd,    \
                     hd_out)
  if (q_dtype == kF32 && cache_dtype == kF32) ATOMA_QKN(float, float);
  else if (q_dtype == kBF16 && cache_dtype == kBF16) ATOMA_QKN(bf16_t, bf16_t);
  else return ATOMA_ERR_DTYPE;
#undef ATOMA_QKN
  ATOMA_LAUNCH_CHECK();
  return 0;
}
