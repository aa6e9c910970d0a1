// A selective state-space recurrence with one scalar decay per head (the Mamba-2 form): per head and request a
// float32 matrix S [n, vdim] that every token decays, writes and reads,
//
//   S <- a S + dt B x^T;   y = S^T C + D x,        a = exp(-exp(A_log) dt),  dt = softplus(dt_raw + dt_bias),
//
// with x (vdim per head), B and C (n per group of heads) the token's projections after a short causal convolution over
// time (with bias) and SiLU.  Everything here is float32.  Its kernels:
//   ssd_prepare      per token: the convolution (the taps - 1 inputs before an entry's first token come from the
//                    request's state), bias and SiLU of the x, B, C channels; dt and the decay of every head;
//   ssd_conv_state   per request: the last taps - 1 inputs of the convolution, for the request's next step;
//   ssd_scan         per (request, head, 16 columns of S): the recurrence over the entry's tokens in order, S read from
//                    the request's state slot before and written back after.  A column of S lives in the registers of
//                    16 neighbouring lanes (n / 16 rows each, rounded up); the tokens' inputs pass LDS in blocks;
//   ssd_scores,      the same recurrence for entries of many tokens (prompts and their portions), 64 tokens at a time on
//   ssd_chunk        the matrix cores in float32 (v_mfma_f32_16x16x4_f32), see below;
//   ssd_step         prepare, conv_state and scan in one, for steps of single tokens;
//   ssd_out          per token and norm group: y * silu(z), divided by the root mean square of its group, times the
//                    weight, in the activation dtype.
// The order of every sum depends on the sizes alone, so a token's result does not depend on how the request was cut
// into steps or on what else the step holds.
//
// State of a request (float32, one row of the state tensor):  [taps - 1][conv channels]  then  [heads][vdim][n].
#include "common.h"

using namespace atoma;

struct SsdShape {
  int heads, groups, vdim, n, taps;
  int ldp;                          // row stride of the projections
  int off_z, off_x, off_dt;         // first columns of z, of the convolved channels (x, B, C) and of dt in a row
};

__device__ __forceinline__ float ssd_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float ssd_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// conv channels: x (heads * vdim), then B (groups * n), then C (the same), as they lie in a row of the projections.
// A workgroup takes TT neighbouring tokens of 256 channels.  With up to four taps (FEW) it asks for the rows of all of them and the
// three before at once, and only tokens that begin an entry read the state.  Bound by the rows' way to and fro: 2,048 tokens of 4,352
// channels (72 MB) 17.4 us, where a token a workgroup, four conditional loads a channel, took 45.3; of 6,400 channels 24.9 and 64.1; 300
// tokens 5.4 and 9.3, 200 single ones 6.3 and 6.4.  (Eight tokens a workgroup: 16.6, 22.9, 5.8, 7.8.)
template <int TT, bool FEW>
__global__ void __launch_bounds__(256)
ssd_prepare_kernel(const float* __restrict__ proj, SsdShape sh, const int32_t* __restrict__ token_seq,
                   const int32_t* __restrict__ q_start, const int32_t* __restrict__ state_slots,
                   const float* __restrict__ state, size_t state_stride, const float* __restrict__ taps_w,
                   const float* __restrict__ conv_bias, const float* __restrict__ dt_bias,
                   const float* __restrict__ a_log, float* __restrict__ xbc, float* __restrict__ dt,
                   float* __restrict__ decay, int n_tokens) {
  const int t0 = blockIdx.x * TT, tokens = min(TT, n_tokens - t0);
  const int channels = sh.heads * sh.vdim + 2 * sh.groups * sh.n;
  if (blockIdx.y == gridDim.y - 1) {
    // the tokens' last workgroup: step sizes and decays, which need nothing of the convolution
    for (int i = threadIdx.x; i < tokens * sh.heads; i += 256) {
      const int t = t0 + i / sh.heads, h = i % sh.heads;
      const float d = ssd_softplus(proj[(size_t)t * sh.ldp + sh.off_dt + h] + dt_bias[h]);
      dt[(size_t)t * sh.heads + h] = d;
      decay[(size_t)t * sh.heads + h] = expf(-expf(a_log[h]) * d);
    }
    return;
  }
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= channels) return;
  const float bias = conv_bias[c];
  const float* const in = proj + sh.off_x + c;
  if constexpr (FEW) {
    float x[TT + 3], w[4];       // (tap j of `taps` is w[4 - taps + j])
#pragma unroll
    for (int j = 0; j < TT + 3; ++j) x[j] = in[(size_t)min(max(t0 - 3 + j, 0), n_tokens - 1) * sh.ldp];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = taps_w[(size_t)c * sh.taps + max(j - (4 - sh.taps), 0)];
#pragma unroll
    for (int k = 0; k < TT; ++k) {
      if (k >= tokens) break;
      const int t = t0 + k, e = token_seq[t], i = t - q_start[e];
      float y = bias;
      if (i >= sh.taps - 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) y = j >= 4 - sh.taps ? fmaf(w[j], x[k + j], y) : y;
      } else {
        const float* const conv_state = state + (size_t)state_slots[e] * state_stride;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (j < 4 - sh.taps) continue;
          const int s = i - 3 + j;      // index inside the entry of the input under the tap
          y = fmaf(w[j], s >= 0 ? x[k + j] : conv_state[(size_t)(sh.taps - 1 + s) * channels + c], y);
        }
      }
      xbc[(size_t)t * channels + c] = y * ssd_sigmoid(y);
    }
  } else {
    for (int t = t0; t < t0 + tokens; ++t) {
      const int e = token_seq[t], i = t - q_start[e];
      const float* const conv_state = state + (size_t)state_slots[e] * state_stride;
      float y = bias;
      for (int j = 0; j < sh.taps; ++j) {
        const int s = i - (sh.taps - 1) + j;
        const float x = s >= 0 ? in[(size_t)(t - (sh.taps - 1) + j) * sh.ldp] : conv_state[(size_t)(sh.taps - 1 + s) * channels + c];
        y = fmaf(taps_w[(size_t)c * sh.taps + j], x, y);
      }
      xbc[(size_t)t * channels + c] = y * ssd_sigmoid(y);
    }
  }
}

// one thread a (entry, channel): the state's rows in ascending order, so that a row is read before it is overwritten
__global__ void __launch_bounds__(256)
ssd_conv_state_kernel(const float* __restrict__ proj, SsdShape sh, const int32_t* __restrict__ q_start,
                      const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride) {
  const int e = blockIdx.y;
  const int channels = sh.heads * sh.vdim + 2 * sh.groups * sh.n;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= channels) return;
  const int first = q_start[e], count = q_start[e + 1] - first;
  float* st = state + (size_t)state_slots[e] * state_stride;
  const int keep = sh.taps - 1;
  for (int r = 0; r < keep; ++r) {
    const int s = count - keep + r;     // index inside the entry of the input that row r holds afterwards
    st[(size_t)r * channels + c] = s >= 0 ? proj[(size_t)(first + s) * sh.ldp + sh.off_x + c]
                                          : st[(size_t)(r + count) * channels + c];
  }
}

constexpr int kScanTokens = 16;      // tokens whose inputs wait in LDS at a time
constexpr int kScanCols = 16;        // columns of S a workgroup owns

// Sum over 16 neighbouring lanes; every lane gets the same sum (the pairs of each step add the same two numbers).
__device__ __forceinline__ float lanes16_sum(float x) {
  x += __shfl_xor(x, 1, 64);
  x += __shfl_xor(x, 2, 64);
  x += __shfl_xor(x, 4, 64);
  x += __shfl_xor(x, 8, 64);
  return x;
}

// R: rows of S a lane holds; lane l of a column owns rows l, l + 16, l + 32, ...
template <int R>
__global__ void __launch_bounds__(256)
ssd_scan_kernel(const float* __restrict__ xbc, const float* __restrict__ dt, const float* __restrict__ decay,
                const float* __restrict__ d_skip, SsdShape sh, const int32_t* __restrict__ q_start,
                const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride,
                float* __restrict__ y, int below) {
  __shared__ float sb[kScanTokens][16 * R], sc[kScanTokens][16 * R];
  __shared__ float sx[kScanTokens][kScanCols], sdt[kScanTokens], sa[kScanTokens];
  const int e = blockIdx.z, h = blockIdx.y, v0 = blockIdx.x * kScanCols;
  const int first = q_start[e], count = q_start[e + 1] - first;
  if (count <= 0 || count >= below) return;      // (entries of `below` tokens or more are the chunk kernel's)
  const int col = threadIdx.x >> 4, l = threadIdx.x & 15;
  const int v = v0 + col;
  const bool live = v < sh.vdim;
  const int inner = sh.heads * sh.vdim, gn = sh.groups * sh.n, channels = inner + 2 * gn;
  const int g = h / (sh.heads / sh.groups);
  float* s_ptr = state + (size_t)state_slots[e] * state_stride + (size_t)(sh.taps - 1) * channels +
                 ((size_t)h * sh.vdim + (live ? v : 0)) * sh.n;
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int row = l + 16 * r;
    s[r] = (live && row < sh.n) ? s_ptr[row] : 0.f;
  }
  const float dh = d_skip[h];
  for (int t0 = 0; t0 < count; t0 += kScanTokens) {
    const int nt = count - t0 < kScanTokens ? count - t0 : kScanTokens;
    __syncthreads();
    for (int idx = threadIdx.x; idx < nt * 16 * R; idx += 256) {
      const int tt = idx / (16 * R), row = idx % (16 * R);
      const size_t base = (size_t)(first + t0 + tt) * channels + inner + (size_t)g * sh.n;
      sb[tt][row] = row < sh.n ? xbc[base + row] : 0.f;
      sc[tt][row] = row < sh.n ? xbc[base + gn + row] : 0.f;
    }
    for (int idx = threadIdx.x; idx < nt * kScanCols; idx += 256) {
      const int tt = idx / kScanCols, cc = idx % kScanCols;
      sx[tt][cc] = v0 + cc < sh.vdim ? xbc[(size_t)(first + t0 + tt) * channels + (size_t)h * sh.vdim + v0 + cc] : 0.f;
    }
    if (threadIdx.x < nt) {
      sdt[threadIdx.x] = dt[(size_t)(first + t0 + threadIdx.x) * sh.heads + h];
      sa[threadIdx.x] = decay[(size_t)(first + t0 + threadIdx.x) * sh.heads + h];
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float a = sa[tt], xv = sx[tt][col], w = sdt[tt] * xv;
      float acc = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[r] = fmaf(a, s[r], w * sb[tt][l + 16 * r]);
        acc = fmaf(s[r], sc[tt][l + 16 * r], acc);
      }
      acc = lanes16_sum(acc);
      if (l == 0 && live) y[(size_t)(first + t0 + tt) * inner + (size_t)h * sh.vdim + v] = acc + dh * xv;
    }
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = l + 16 * r;
      if (row < sh.n) s_ptr[row] = s[r];
    }
  }
}

// A step of single tokens (every entry has one): prepare, convolution state and scan in one launch, a workgroup a (request, head,
// 16 * PASSES columns of S).  The columns are asked for before anything else and arrive while the workgroup makes the convolution of
// its x and, as every head of a group does, of the group's B and C; the sums are added as above: the same bits.  x's part of the
// convolution's state belongs to one workgroup, which replaces it; B's and C's, which all heads of the group read, are left to
// ssd_out.  Bound by the state's bytes, from two trips to memory on.  Eight requests of 64 heads of 128 x 64 (34 MB
// read and written): 10.3 us, where prepare, the convolution's state and the scan take 5.0 + 5.2 + 8.5; 21 with masks on the state at
// its loads, which the compiler then waits for one by one.
template <int R, int PASSES>
__global__ void __launch_bounds__(256)
ssd_step_kernel(const float* __restrict__ proj, SsdShape sh, const int32_t* __restrict__ q_start,
                const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride,
                const float* __restrict__ taps_w, const float* __restrict__ conv_bias, const float* __restrict__ dt_bias,
                const float* __restrict__ a_log, const float* __restrict__ d_skip, float* __restrict__ y) {
  constexpr int COLS = 16 * PASSES;
  __shared__ float sb[16 * R], sc[16 * R], sx[COLS], scalars[3];
  const int e = blockIdx.z, h = blockIdx.y, v0 = blockIdx.x * COLS, tid = threadIdx.x;
  const int inner = sh.heads * sh.vdim, gn = sh.groups * sh.n, channels = inner + 2 * gn, keep = sh.taps - 1;
  const int g = h / (sh.heads / sh.groups), col = tid >> 4, l = tid & 15;
  const int t = q_start[e];
  float* const st = state + (size_t)state_slots[e] * state_stride;
  float* const sp = st + (size_t)keep * channels + ((size_t)h * sh.vdim + v0) * sh.n;
  const int live = min(COLS, sh.vdim - v0);         // columns that exist
  float s[PASSES][R];
#pragma unroll
  for (int p = 0; p < PASSES; ++p)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int v = p * 16 + col, row = l + 16 * r;
      s[p][r] = sp[(uint32_t)(min(v, live - 1) * sh.n + min(row, sh.n - 1))];
    }
  auto input = [&](int c) { return proj[(size_t)t * sh.ldp + sh.off_x + c]; };
  float held[4] = {0.f, 0.f, 0.f, 0.f}, held_in = 0.f;      // of the thread's column of x: the earlier inputs and the token's
  static_assert(COLS <= 256, "x is everybody's first channel");
  for (int i = tid; i < COLS + 32 * R; i += 256) {
    const int j = (i - COLS) % (16 * R);
    const bool of_c = i >= COLS + 16 * R, there = i < COLS ? i < live : j < sh.n;
    float out = 0.f;
    if (there) {
      const int c = i < COLS ? h * sh.vdim + v0 + i : inner + (of_c ? gn : 0) + g * sh.n + j;
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      const float in = input(c), z = convolve_one(st + c, taps_w + (size_t)c * sh.taps, keep, channels, in, conv_bias[c], x);
      out = z * ssd_sigmoid(z);
      if (i == tid) {
        held_in = in;
#pragma unroll
        for (int q = 0; q < 4; ++q) held[q] = x[q];
      }
    }
    (i < COLS ? sx + i : of_c ? sc + j : sb + j)[0] = out;
  }
  // (one lane, of a wave whose others have no second channel: its trip to memory runs beside theirs)
  if (tid == 255) {
    const float rate = expf(a_log[h]), step = ssd_softplus(proj[(size_t)t * sh.ldp + sh.off_dt + h] + dt_bias[h]);
    scalars[0] = step, scalars[1] = expf(-rate * step), scalars[2] = d_skip[h];
  }
  lds_barrier();
  const float d = scalars[0], a = scalars[1], dh = scalars[2];
  float b[R], cc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) b[r] = sb[l + 16 * r], cc[r] = sc[l + 16 * r];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int v = p * 16 + col;
    const float xv = sx[v], w = d * xv;
    float acc = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // (made zero here and not at the load, which would then stand under the condition and be waited for at once)
      s[p][r] = l + 16 * r < sh.n ? fmaf(a, s[p][r], w * b[r]) : 0.f;
      acc = fmaf(s[p][r], cc[r], acc);
    }
    acc = lanes16_sum(acc);
    if (v < live) {
      if (l == 0) y[(size_t)t * inner + (size_t)h * sh.vdim + v0 + v] = acc + dh * xv;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (l + 16 * r < sh.n) sp[(size_t)v * sh.n + l + 16 * r] = s[p][r];
    }
  }
  if (tid < live) push_inputs(st + h * sh.vdim + v0 + tid, keep, channels, held_in, held, true);
}

// The recurrence 64 tokens at a time.  With c_t the sum of the log decays of the chunk's tokens up to t (inclusive),
//   y_t = sum_{s <= t} exp(c_t - c_s) dt_s (C_t . B_s) x_s  +  exp(c_t) S_0^T C_t  +  D x_t,
//   S_64 = exp(c_63) S_0 + sum_s exp(c_63 - c_s) dt_s B_s x_s^T,
// every exponent at most zero.  The products C_t . B_s are the same for all heads of a group and all columns of S: a
// first kernel (ssd_scores) makes them once per (chunk, group).  Then a workgroup owns (entry, head, 16 columns of S)
// and walks the entry's chunks in order; per chunk each of its four waves takes 16 tokens of y = M X + diag(exp(c)) C S, with
// M[t][s] = (C_t . B_s) exp(c_t - c_s) dt_s for s <= t, then its share of the rows of S.
// All products are float32 MFMAs of 16 x 16 x 4 (result D[4 (l / 16) + i][l % 16] in lane l).  The sum over k of a
// block of 16 is taken in the order that lets a lane have its four values as one 16-byte piece: in the block's MFMA j, lane l
// gives A[l % 16][4 (l / 16) + j] and B[4 (l / 16) + j][l % 16].  C's and B's rows and the tiles of scores come from memory as
// the operands that they are, each of them to the one wave that multiplies it, and M is made of the scores in registers; a wave's
// rows of S stay in its registers too.  What the waves share passes LDS, transposed for the pieces, in two buffers that take turns:
// x, and S for y.  So a chunk has one barrier, and each operand is asked for as soon as the one before it has been used.
// Bound by a wave's way through a chunk, 3.7 us with a state of 128, of which its 36 to 48 MFMAs for y and 32 for S are 1.1, and where
// entries are many by all waves' instructions; it was 6 us, with five barriers and all operands through 108 KB of LDS, one workgroup a CU.
// us with the scores, before / now: 64 heads of 64 x 128, one entry of 2,048 tokens 202 / 114, 1,400 and 640 206 / 95, eight of 256 229 / 98,
// 64 of 32 598 / 212; 32 heads of 64 x 64, one of 2,048 143 / 87.  The results' bits are the same.  (The next chunk's sums of decays made
// between this one's MFMAs, or B's rows by pairs, gave nothing: 139 and 135 against 136 at that point.)
constexpr int kChunk = 64;
constexpr int kChunkLdt = kChunk + 4;      // row stride of x transposed
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

#if defined(__HIP_DEVICE_COMPILE__)
__device__ __forceinline__ auto buffer(const float* p, int floats) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, __builtin_amdgcn_readfirstlane(floats * 4), 0x00027000);
}
template <typename B>
__device__ __forceinline__ float one(B from, uint32_t at) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0));
}
template <typename B>
__device__ __forceinline__ f32x4 four(B from, uint32_t at) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
}
// the place of float `at`, or one that is out of any buffer's range and comes as zero (which stays a value of a register: known to be a
// constant, it becomes a branch around the load)
__device__ __forceinline__ uint32_t place(bool in, int at) {
  uint32_t x = in ? (uint32_t)at * 4 : 0x80000000u;
  asm("" : "+v"(x));
  return x;
}
// a row's NB blocks of 16 columns from `row` on, of which the lane has 4 (l / 16) .. + 3; `last`: the places in the last block, which alone
// can end early
template <int NB, bool VEC, typename B>
__device__ __forceinline__ void operand(B from, int row, const uint32_t (&last)[4], f32x4 (&x)[NB]) {
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if constexpr (VEC) {
      x[b] = four(from, b < NB - 1 ? (uint32_t)(row + b * 16) * 4 : last[0]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) x[b][q] = one(from, b < NB - 1 ? (uint32_t)(row + b * 16 + q) * 4 : last[q]);
    }
  }
}
template <int NB, bool VEC>
__device__ __forceinline__ void last_places(int row, int column, int n, uint32_t (&last)[4]) {
#pragma unroll
  for (int q = 0; q < (VEC ? 1 : 4); ++q) last[q] = place((NB - 1) * 16 + column + q < n, row + (NB - 1) * 16 + q);
}
#endif

// VEC: C and S are fetched 16 bytes at a time (state size, channel counts and the state's rows all multiples of 4)
template <int NB, bool VEC>      // NB: blocks of 16 rows of S (the state size rounded up)
__global__ void __launch_bounds__(256)
ssd_chunk_kernel(const float* __restrict__ xbc, const float* __restrict__ dt, const float* __restrict__ a_log,
                 const float* __restrict__ d_skip, SsdShape sh, const int32_t* __restrict__ q_start,
                 const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride,
                 float* __restrict__ y, int at_least, const float* __restrict__ scores, int max_chunks) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NP = 16 * NB, LDN = NP + 4, MINE = (NB + 3) / 4;      // MINE: blocks of 16 rows of S of a wave
  __shared__ __attribute__((aligned(16))) float St[2][16 * LDN];          // S transposed: [column][row], as the state keeps it
  __shared__ __attribute__((aligned(16))) float Xt[2][16 * kChunkLdt];    // x transposed: [column][token]
  __shared__ __attribute__((aligned(16))) float own[4][3][kChunk];        // of a wave: log decays summed up to a token, dt, and
                                                                          // exp(c_last - c_s) dt_s
  const int e = blockIdx.z, h = blockIdx.y, v0 = blockIdx.x * 16;
  const int first = q_start[e], count = q_start[e + 1] - first;
  if (count < at_least) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int inner = sh.heads * sh.vdim, gn = sh.groups * sh.n, channels = inner + 2 * gn;
  const int g = h / (sh.heads / sh.groups);
  const int vlive = min(16, sh.vdim - v0);
  const float rate = expf(a_log[h]), dh = d_skip[h];
  float* const cum = own[wave][0];
  float* const dts = own[wave][1];
  float* const wts = own[wave][2];

  // a chunk's rows of xbc, of dt and of scores; past the last chunk nothing is in range.  (No load stands under a condition, which the
  // compiler would wait for where the branches meet.)
  auto rows_of = [&](int t0) { return max(0, min(kChunk, count - t0)); };
  auto inputs = [&](int t0) { return buffer(xbc + (size_t)(first + t0) * channels, rows_of(t0) * channels); };
  const uint32_t x_at = place((tid & 15) < vlive, (tid >> 4) * channels + h * sh.vdim + v0 + (tid & 15));
  const uint32_t y_at = place(r16 < vlive, (wave * 16 + 4 * kg) * inner + r16);
  const int c_row = (wave * 16 + r16) * channels + inner + gn + g * sh.n + 4 * kg;
  uint32_t c_last[4], b_at[MINE], mt_at[4];
  last_places<NB, VEC>(c_row, 4 * kg, sh.n, c_last);
#pragma unroll
  for (int m = 0; m < MINE; ++m) {
    const int n = (wave + 4 * m) * 16 + r16;
    b_at[m] = place(n < sh.n, 4 * kg * channels + inner + g * sh.n + n);
  }
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) mt_at[sb] = place(sb <= wave, ((wave * (wave + 1) / 2 + sb) * 64 + lane) * 4);
  f32x4 cc[NB], mt[4];
  float bb[MINE][4][4], rx[4], rdt;
  auto fetch_x = [&](int t0) {
    const auto from = inputs(t0);
#pragma unroll
    for (int i = 0; i < 4; ++i) rx[i] = one(from, x_at + (uint32_t)(i * 16 * channels) * 4);
    const int rows = rows_of(t0);
    rdt = one(buffer(dt + (size_t)(first + t0) * sh.heads + h, rows > 0 ? (rows - 1) * sh.heads + 1 : 0), (uint32_t)(lane * sh.heads) * 4);
  };
  // C's rows of the wave's 16 tokens, and its tiles of scores
  auto fetch_c = [&](int t0) {
    operand<NB, VEC>(inputs(t0), c_row, c_last, cc);
    const auto tiles = buffer(scores + (((size_t)e * max_chunks + t0 / kChunk) * sh.groups + g) * (10 * 256), rows_of(t0) > 0 ? 10 * 256 : 0);
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
      mt[sb] = four(tiles, mt_at[sb]);
  };
  // B's columns that are the wave's rows of S
  auto fetch_b = [&](int t0) {
    const auto from = inputs(t0);
#pragma unroll
    for (int m = 0; m < MINE; ++m)
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) bb[m][k][q] = one(from, b_at[m] + (uint32_t)((k * 16 + q) * channels) * 4);
  };
  auto stash_x = [&](float* xt) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + i * 256;
      xt[(idx & 15) * kChunkLdt + (idx >> 4)] = rx[i];
    }
  };

  fetch_x(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_c(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_b(0);
  __builtin_amdgcn_sched_barrier(0);
  // lane: rows (wave + 4 m) 16 + 4 (l / 16) .. + 3 of S, column l % 16
  float* const s_ptr = state + (size_t)state_slots[e] * state_stride + (size_t)(sh.taps - 1) * channels +
                       ((size_t)h * sh.vdim + v0 + min(r16, vlive - 1)) * sh.n;
  f32x4 s[MINE];
#pragma unroll
  for (int m = 0; m < MINE; ++m) {
    const int n = (wave + 4 * m) * 16 + 4 * kg;
    s[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (VEC) {
      if (r16 < vlive && n < sh.n) s[m] = *reinterpret_cast<const f32x4*>(s_ptr + n);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (r16 < vlive && n + q < sh.n) s[m][q] = s_ptr[n + q];
    }
    if (wave + 4 * m < NB) *reinterpret_cast<f32x4*>(St[0] + r16 * LDN + n) = s[m];
  }
  stash_x(Xt[0]);
  __syncthreads();
  for (int t0 = 0; t0 < count; t0 += kChunk) {
    const int nt = min(kChunk, count - t0), buf = (t0 / kChunk) & 1;
    const size_t tok0 = (size_t)(first + t0);
    // inclusive sums of the log decays over the 64 lanes
    float c = -rate * rdt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float up = __shfl_up(c, o, 64);
      if (lane >= o) c += up;
    }
    const float last = __shfl(c, 63, 64), ec = expf(c);
    cum[lane] = c;
    dts[lane] = rdt;
    wts[lane] = expf(last - c) * rdt;
    const float keep = __shfl(ec, 63, 64), et = __shfl(ec, wave * 16 + r16, 64), ct = __shfl(c, wave * 16 + r16, 64);
    __builtin_amdgcn_wave_barrier();      // (what is read of it below was written by this wave)
    const float* const xp = Xt[buf] + r16 * kChunkLdt + 4 * kg;
    fetch_x(t0 + kChunk);
    __builtin_amdgcn_sched_barrier(0);
    // y of the wave's 16 tokens
    if (wave * 16 < nt) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
      const f32x4 x4 = lds4(xp + wave * 16);
#pragma unroll
      for (int sb = 0; sb < 4; ++sb) {
        if (sb > wave) continue;
        const f32x4 cs = lds4(cum + sb * 16 + 4 * kg), ds = lds4(dts + sb * 16 + 4 * kg), b4 = lds4(xp + sb * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float m = mt[sb][q] * expf(ct - cs[q]) * ds[q];
          asm("" : "+v"(m));      // (it is not worth a branch)
          if (sb == wave && 4 * kg + q > r16) m = 0.f;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(m, b4[q], acc, 0, 0, 0);
        }
      }
      const float* const sp = St[buf] + r16 * LDN + 4 * kg;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const f32x4 b4 = lds4(sp + b * 16);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(et * cc[b][q], b4[q], acc, 0, 0, 0);
      }
      const auto to = buffer(y + tok0 * inner + (size_t)h * sh.vdim + v0, (nt - 1) * inner + vlive);      // (what is out of range stays unwritten)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i] + dh * x4[i]), to, y_at + (uint32_t)(i * inner) * 4, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);      // (the loads arrive in the order in which they are asked for)
    fetch_c(t0 + kChunk);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MINE; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[m][i] *= keep;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 w4 = lds4(wts + k * 16 + 4 * kg), b4 = lds4(xp + k * 16);
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int m = 0; m < MINE; ++m) s[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb[m][k][q] * w4[q], b4[q], s[m], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    fetch_b(t0 + kChunk);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MINE; ++m)
      if (wave + 4 * m < NB) *reinterpret_cast<f32x4*>(St[buf ^ 1] + r16 * LDN + (wave + 4 * m) * 16 + 4 * kg) = s[m];
    stash_x(Xt[buf ^ 1]);
    __syncthreads();       // the next chunk's x and S are there, and everybody is done with this one's
  }
#pragma unroll
  for (int m = 0; m < MINE; ++m) {
    const int n = (wave + 4 * m) * 16 + 4 * kg;
    if constexpr (VEC) {
      if (r16 < vlive && n < sh.n) *reinterpret_cast<f32x4*>(s_ptr + n) = s[m];
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (r16 < vlive && n + q < sh.n) s_ptr[n + q] = s[m][q];
    }
  }
#endif
}

// C_t . B_s of every chunk of 64 tokens, once per group of heads: the ten 16 x 16 tiles on and below the diagonal, each
// as its 64 lanes' four numbers (lane l: t = l % 16, s = 4 (l / 16) .. + 3 of the tile, as M's operand wants them),
// [entry][chunk][group][10][64][4].  A wave a tile, its operands straight from memory: one trip there and 4 NB MFMAs.  (2,048 tokens, a
// state of 128: some 5 us; a workgroup a chunk, which took B and C to LDS first, 20.)
template <int NB, bool VEC>
__global__ void __launch_bounds__(256)
ssd_scores_kernel(const float* __restrict__ xbc, SsdShape sh, const int32_t* __restrict__ q_start, int at_least,
                  float* __restrict__ scores, int max_chunks) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, kg = lane >> 4;
  const int chunk = blockIdx.x / 3, j = blockIdx.x % 3 * 4 + wave, e = blockIdx.z, g = blockIdx.y, t0 = chunk * kChunk;
  const int first = q_start[e], count = q_start[e + 1] - first;
  if (count < at_least || t0 >= count || j >= 10) return;
  const int tb = j >= 6 ? 3 : j >= 3 ? 2 : j >= 1 ? 1 : 0, sb = j - tb * (tb + 1) / 2;
  const int inner = sh.heads * sh.vdim, gn = sh.groups * sh.n, channels = inner + 2 * gn;
  const auto from = buffer(xbc + (size_t)(first + t0) * channels, min(kChunk, count - t0) * channels);
  const int b_row = (sb * 16 + r16) * channels + inner + g * sh.n + 4 * kg, c_row = (tb * 16 + r16) * channels + inner + gn + g * sh.n + 4 * kg;
  uint32_t b_last[4], c_last[4];
  last_places<NB, VEC>(b_row, 4 * kg, sh.n, b_last);
  last_places<NB, VEC>(c_row, 4 * kg, sh.n, c_last);
  f32x4 bb[NB], cc[NB], acc = f32x4{0.f, 0.f, 0.f, 0.f};
  operand<NB, VEC>(from, b_row, b_last, bb);
  operand<NB, VEC>(from, c_row, c_last, cc);
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bb[b][q], cc[b][q], acc, 0, 0, 0);
  *reinterpret_cast<f32x4*>(scores + ((((size_t)e * max_chunks + chunk) * sh.groups + g) * 10 + j) * 256 + lane * 4) = acc;
#endif
}

// What is left of the convolution's state after ssd_step_kernel (state: null elsewhere): channels from `first` on of the token's request
struct SsdTail {
  float* state;
  const int32_t* state_slots;
  size_t stride;
  int off_x, first, channels, keep;
};

// one workgroup per (token, norm group); parts of up to 4,096 columns wait in registers between the two passes.  A thread does the work
// of V threads of a block of V * NT, sums apart, so that a row's result is the same whatever V: few rows want many threads (eight tokens of
// 4,096 columns 5.1 us with 1,024 threads, 6.8 with 256), many rows fewer, since a CU then has more rows on their way.
template <typename TO, int PER, int NT, int V, bool TAIL>
__global__ void __launch_bounds__(NT)
ssd_out_kernel(const float* __restrict__ y, const float* __restrict__ proj, int ldp, int off_z,
               const float* __restrict__ w, float eps, int inner, int part, TO* __restrict__ out, SsdTail tail) {
  constexpr int WAVES = NT / 64;
  __shared__ float scratch[WAVES * V];
  const int t = blockIdx.x, p0 = blockIdx.y * part;
  if (TAIL && blockIdx.y == 0) {
    // (a step of single tokens: token t is entry t's)
    float* const st = tail.state + (size_t)tail.state_slots[t] * tail.stride;
    for (int c = tail.first + threadIdx.x; c < tail.channels; c += NT) {
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = st[(size_t)min(r, tail.keep - 1) * tail.channels + c];
      push_inputs(st + c, tail.keep, tail.channels, proj[(size_t)t * ldp + tail.off_x + c], x, true);
    }
  }
  const float* zp = proj + (size_t)t * ldp + off_z + p0;
  const float* yp = y + (size_t)t * inner + p0;
  float ss[V];
#pragma unroll
  for (int q = 0; q < V; ++q) ss[q] = 0.f;
  // over the threads of the block of V * NT, in their order
  auto sum = [&]() {
    if constexpr (V == 1) return block_sum<WAVES>(ss[0], scratch);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const float all = wave_sum(ss[q]);
      if (lane == 0) scratch[q * WAVES + wave] = all;
    }
    lds_barrier();
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES * V; ++i) total += scratch[i];
    return total;
  };
  if constexpr (PER > 0) {
    constexpr int P = PER * V;
    float u[P], yv[P], zv[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const int i = threadIdx.x + j * NT;
      yv[j] = i < part ? yp[i] : 0.f;
      zv[j] = i < part ? zp[i] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < P; ++j) {
      u[j] = yv[j] * (zv[j] * ssd_sigmoid(zv[j]));
      ss[j % V] = fmaf(u[j], u[j], ss[j % V]);
    }
    const float inv = 1.0f / sqrtf(sum() / (float)part + eps);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const int i = threadIdx.x + j * NT;
      if (i < part) out[(size_t)t * inner + p0 + i] = from_f32<TO>(u[j] * inv * w[p0 + i]);
    }
    return;
  }
  static_assert(PER > 0 || V == 1, "a row that is walked twice: a thread an own sum");
  for (int i = threadIdx.x; i < part; i += NT) {
    const float z = zp[i];
    const float u = yp[i] * (z * ssd_sigmoid(z));
    ss[0] = fmaf(u, u, ss[0]);
  }
  const float inv = 1.0f / sqrtf(sum() / (float)part + eps);
  for (int i = threadIdx.x; i < part; i += NT) {
    const float z = zp[i];
    const float u = yp[i] * (z * ssd_sigmoid(z));
    out[(size_t)t * inner + p0 + i] = from_f32<TO>(u * inv * w[p0 + i]);
  }
}

static bool shape_ok(const SsdShape& sh) {
  return sh.heads > 0 && sh.groups > 0 && sh.heads % sh.groups == 0 && sh.vdim > 0 && sh.n > 0 && sh.n <= 256 &&
         sh.taps >= 1 && sh.taps <= 64 && sh.ldp > 0 && sh.off_z >= 0 && sh.off_x >= 0 && sh.off_dt >= 0;
}

extern "C" int atoma_ssd_prepare(const float* proj, int ldp, int off_z, int off_x, int off_dt, int heads, int groups,
                                 int vdim, int n, int taps, const int32_t* token_seq, const int32_t* q_start,
                                 const int32_t* state_slots, const float* state, size_t state_stride,
                                 const float* taps_w, const float* conv_bias, const float* dt_bias,
                                 const float* a_log, float* xbc, float* dt, float* decay, int n_tokens,
                                 hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  SsdShape sh{heads, groups, vdim, n, taps, ldp, off_z, off_x, off_dt};
  if (!shape_ok(sh)) return ATOMA_ERR_SHAPE;
  const int channels = heads * vdim + 2 * groups * n;
  const int blocks = (channels + 255) / 256 + 1;
  if (blocks > 65535) return ATOMA_ERR_SHAPE;
#define ATOMA_PREPARE(TT, FEW)                                                                                                      \
  hipLaunchKernelGGL((ssd_prepare_kernel<TT, FEW>), dim3((n_tokens + TT - 1) / TT, blocks), dim3(256), 0, stream, proj, sh, token_seq,  \
                     q_start, state_slots, state, state_stride, taps_w, conv_bias, dt_bias, a_log, xbc, dt, decay, n_tokens)
  // (single tokens, each an entry of its own, would read the state four times one after the other: up to some hundred nothing is gained)
  if (taps <= 4 && n_tokens >= 128) ATOMA_PREPARE(4, true);
  else ATOMA_PREPARE(1, false);
#undef ATOMA_PREPARE
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_ssd_conv_state(const float* proj, int ldp, int off_x, int heads, int groups, int vdim, int n,
                                    int taps, const int32_t* q_start, const int32_t* state_slots, float* state,
                                    size_t state_stride, int n_entries, hipStream_t stream) {
  if (n_entries <= 0 || taps <= 1) return 0;
  SsdShape sh{heads, groups, vdim, n, taps, ldp, 0, off_x, 0};
  if (!shape_ok(sh) || n_entries > 65535) return ATOMA_ERR_SHAPE;
  const int channels = heads * vdim + 2 * groups * n;
  hipLaunchKernelGGL(ssd_conv_state_kernel, dim3((channels + 255) / 256, n_entries), dim3(256), 0, stream, proj, sh,
                     q_start, state_slots, state, state_stride);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_ssd_scan(const float* xbc, const float* dt, const float* decay, const float* d_skip, int heads,
                              int groups, int vdim, int n, int taps, const int32_t* q_start,
                              const int32_t* state_slots, float* state, size_t state_stride, float* y,
                              int n_entries, int below, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  SsdShape sh{heads, groups, vdim, n, taps, 1, 0, 0, 0};
  if (!shape_ok(sh) || n_entries > 65535 || heads > 65535) return ATOMA_ERR_SHAPE;
  dim3 grid((vdim + kScanCols - 1) / kScanCols, heads, n_entries), block(256);
  const int rows = (n + 15) / 16;
#define ATOMA_SCAN(R)                                                                                              \
  hipLaunchKernelGGL((ssd_scan_kernel<R>), grid, block, 0, stream, xbc, dt, decay, d_skip, sh, q_start, state_slots, \
                     state, state_stride, y, below)
  if (rows <= 1) ATOMA_SCAN(1);
  else if (rows <= 2) ATOMA_SCAN(2);
  else if (rows <= 3) ATOMA_SCAN(3);
  else if (rows <= 4) ATOMA_SCAN(4);
  else if (rows <= 6) ATOMA_SCAN(6);
  else if (rows <= 8) ATOMA_SCAN(8);
  else if (rows <= 12) ATOMA_SCAN(12);
  else ATOMA_SCAN(16);
#undef ATOMA_SCAN
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// The largest state size the chunk kernel is built for: a lane has a chunk's operands and its share of S in registers, 32 numbers of C, 32 of B
// and 8 of S at 128.  LDS has room for more; nothing has been measured beyond.
extern "C" int atoma_ssd_chunk_max_state() { return 128; }

template <int NB, bool VEC>
static int launch_chunk(dim3 grid, hipStream_t stream, const float* xbc, const float* dt, const float* a_log,
                        const float* d_skip, const SsdShape& sh, const int32_t* q_start, const int32_t* state_slots,
                        float* state, size_t state_stride, float* y, int at_least, float* scores, int max_chunks) {
  hipLaunchKernelGGL((ssd_scores_kernel<NB, VEC>), dim3(3 * max_chunks, sh.groups, grid.z), dim3(256), 0, stream, xbc, sh,
                     q_start, at_least, scores, max_chunks);
  hipLaunchKernelGGL((ssd_chunk_kernel<NB, VEC>), grid, dim3(256), 0, stream, xbc, dt, a_log, d_skip, sh, q_start,
                     state_slots, state, state_stride, y, at_least, scores, max_chunks);
  return 0;
}

// Floats of scratch that atoma_ssd_chunk needs for entries of up to `max_chunks` chunks of 64 tokens.
extern "C" size_t atoma_ssd_chunk_scratch_floats(int n_entries, int max_chunks, int groups) {
  return (size_t)n_entries * max_chunks * groups * 10 * 256;
}

// entries of at least `at_least` tokens; the others are left to atoma_ssd_scan(below = at_least).  `max_chunks`: chunks
// of 64 tokens of the longest entry; `scores`: scratch of atoma_ssd_chunk_scratch_floats floats.
extern "C" int atoma_ssd_chunk(const float* xbc, const float* dt, const float* a_log, const float* d_skip, int heads,
                               int groups, int vdim, int n, int taps, const int32_t* q_start,
                               const int32_t* state_slots, float* state, size_t state_stride, float* y,
                               int n_entries, int at_least, float* scores, int max_chunks, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  SsdShape sh{heads, groups, vdim, n, taps, 1, 0, 0, 0};
  if (!shape_ok(sh) || n > 128 || n_entries > 65535 || heads > 65535 || groups > 65535 || at_least < 1 ||
      max_chunks < 1 || scores == nullptr)
    return ATOMA_ERR_SHAPE;
  dim3 grid((vdim + 15) / 16, heads, n_entries);
  int rc;
  // (a state size that is a multiple of 4 is then also a whole number of 16-byte pieces of its NB blocks' row)
  const bool vec = n % 4 == 0 && (heads * vdim) % 4 == 0 && state_stride % 4 == 0 && (((uintptr_t)xbc | (uintptr_t)state) & 15) == 0;
#define ATOMA_CHUNK(NB_)                                                                                            \
  rc = vec ? launch_chunk<NB_, true>(grid, stream, xbc, dt, a_log, d_skip, sh, q_start, state_slots, state,        \
                                     state_stride, y, at_least, scores, max_chunks)                               \
           : launch_chunk<NB_, false>(grid, stream, xbc, dt, a_log, d_skip, sh, q_start, state_slots, state,       \
                                      state_stride, y, at_least, scores, max_chunks)
  switch ((n + 15) / 16) {
    case 1: ATOMA_CHUNK(1); break;
    case 2: ATOMA_CHUNK(2); break;
    case 3: ATOMA_CHUNK(3); break;
    case 4: ATOMA_CHUNK(4); break;
    case 5: ATOMA_CHUNK(5); break;
    case 6: ATOMA_CHUNK(6); break;
    case 7: ATOMA_CHUNK(7); break;
    default: ATOMA_CHUNK(8); break;
  }
#undef ATOMA_CHUNK
  if (rc != 0) return rc;
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_ssd_out(const float* y, const float* proj, int ldp, int off_z, const float* w, float eps,
                             int inner, int norm_groups, void* out, int out_dtype, int n_tokens, float* state,
                             const int32_t* state_slots, size_t state_stride, int off_x, int channels, int taps, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (inner <= 0 || norm_groups <= 0 || inner % norm_groups || norm_groups > 65535 || ldp < inner) return ATOMA_ERR_SHAPE;
  const int part = inner / norm_groups;
  if (taps < 2) state = nullptr;
  if (state != nullptr && (channels < inner || state_slots == nullptr || taps > 64)) return ATOMA_ERR_SHAPE;
  const SsdTail tail{state, state_slots, state_stride, off_x, inner, channels, taps - 1};
  const dim3 grid(n_tokens, norm_groups);
#define ATOMA_SSD_OUT_AS(TO, PER, NT, V, TAIL)                                                                                     \
  hipLaunchKernelGGL((ssd_out_kernel<TO, PER, NT, V, TAIL>), grid, dim3(NT), 0, stream, y, proj, ldp, off_z, w, eps, inner, part, \
                     (TO*)out, tail)
#define ATOMA_SSD_OUT(TO, PER, NT, V)                                    \
  do {                                                                   \
    if (state != nullptr) ATOMA_SSD_OUT_AS(TO, PER, NT, V, true);        \
    else ATOMA_SSD_OUT_AS(TO, PER, NT, V, false);                        \
  } while (0)
  // (rows from which on 256 threads are the quicker ones, us by 1,024 / by 256: of 2,048 columns 1,000 10.1 / 10.5, 1,400 13.2 / 12.7,
  // 4,096 31.6 / 25.7; of 3,072 1,400 14.8 / 15.1, 2,048 19.5 / 19.3, 4,096 36.2 / 32.0; longer ones walk the row twice, where 1,024 win or
  // are as quick: of 8,192 512 15.2 / 29.7, 4,096 111 / 113)
  const bool many = (size_t)n_tokens * norm_groups > (part <= 2048 ? 1280 : 1792);
#define ATOMA_SSD_OUT_BY_PART(TO)                                \
  do {                                                           \
    if (part <= 1024) ATOMA_SSD_OUT(TO, 4, 256, 1);              \
    else if (part <= 4096 && many) ATOMA_SSD_OUT(TO, 4, 256, 4); \
    else if (part <= 4096) ATOMA_SSD_OUT(TO, 4, 1024, 1);        \
    else ATOMA_SSD_OUT(TO, 0, 1024, 1);                          \
  } while (0)
  if (out_dtype == kF32) ATOMA_SSD_OUT_BY_PART(float);
  else if (out_dtype == kBF16) ATOMA_SSD_OUT_BY_PART(bf16_t);
  else return ATOMA_ERR_DTYPE;
#undef ATOMA_SSD_OUT_BY_PART
#undef ATOMA_SSD_OUT
#undef ATOMA_SSD_OUT_AS
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// One token of every entry: what atoma_ssd_prepare, atoma_ssd_conv_state and atoma_ssd_scan do in turn, but for B's and C's part of the
// convolution's state, which atoma_ssd_out replaces where it is given the state.
extern "C" int atoma_ssd_step(const float* proj, int ldp, int off_x, int off_dt, int heads, int groups, int vdim, int n, int taps,
                              const int32_t* q_start, const int32_t* state_slots, float* state, size_t state_stride,
                              const float* taps_w, const float* conv_bias, const float* dt_bias, const float* a_log,
                              const float* d_skip, float* y, int n_entries, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  const SsdShape sh{heads, groups, vdim, n, taps, ldp, 0, off_x, off_dt};
  if (!shape_ok(sh) || n_entries > 65535 || heads > 65535) return ATOMA_ERR_SHAPE;
  const int rows = (n + 15) / 16;
#define ATOMA_STEP(R, P)                                                                                                     \
  hipLaunchKernelGGL((ssd_step_kernel<R, P>), dim3((vdim + 16 * P - 1) / (16 * P), heads, n_entries), dim3(256), 0, stream,  \
                     proj, sh, q_start, state_slots, state, state_stride, taps_w, conv_bias, dt_bias, a_log, d_skip, y)
  if (rows <= 1) ATOMA_STEP(1, 4);
  else if (rows <= 2) ATOMA_STEP(2, 4);
  else if (rows <= 3) ATOMA_STEP(3, 4);
  else if (rows <= 4) ATOMA_STEP(4, 4);
  else if (rows <= 6) ATOMA_STEP(6, 4);
  else if (rows <= 8) ATOMA_STEP(8, 4);
  else if (rows <= 12) ATOMA_STEP(12, 2);
  else ATOMA_STEP(16, 2);
#undef ATOMA_STEP
  ATOMA_LAUNCH_CHECK();
  return 0;
}
