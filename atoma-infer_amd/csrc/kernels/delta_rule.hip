// The gated delta rule: a recurrent mixer whose state is one float32 matrix S [dim, vdim] per head and request.
//
// Per token and head (q, k of size dim, unit length; v of size vdim; beta a scalar; g a decay per key channel):
//   S <- diag(g) S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q          (the read-out sees the token's write)
// Everything here is float32.  Four kernels, and delta_step, which does the work of all four for a step of single tokens:
//   delta_prepare      per token: short causal convolution over time and SiLU of the q, k, v projections (the taps - 1
//                      inputs before an entry's first token come from the request's state), q and k to unit length per
//                      head (q also times dim^-1/2), beta = sigmoid(b), g = exp(-exp(A_log) softplus(a + dt_bias));
//   delta_conv_state   per request: the last taps - 1 inputs of the convolution, for the request's next step;
//   delta_scan         per (request, head, 8 or 16 columns of S): the recurrence over the entry's tokens in order, S read
//                      from the request's state slot before and written back after.  A column of S lives in the registers
//                      of 32 or 16 neighbouring lanes, so a token costs a lane a dozen or two multiply-adds and one
//                      exchange of four or six steps among those lanes; the tokens' inputs pass LDS in blocks, fetched a
//                      block ahead;
//   delta_out          per token and head: o / sqrt(mean(o^2) + eps) * w * sigmoid(gate), in the activation dtype.
// The order of every sum depends on the sizes alone, so from the same projections a token's result does not depend on how
// the request was cut into steps or on what else the step holds.  (Float32 projections are the same in any step; those in
// bfloat16 come from a kernel that the step's row count chooses.)
//
// State of a request (float32, one row of the state tensor):  [taps - 1][conv channels]  then  [heads][vdim][dim].
#include <algorithm>

#include "gemm_f32_tile.h"

using namespace atoma;

struct DeltaShape {
  int heads, kv_heads, dim, vdim, taps;
  int ldp;                 // row stride of the projections
  int off_q, off_k, off_v, off_b;   // first columns of the q, k, v and b projections in a row
};

constexpr int kStepThreads = 1024;      // of a workgroup of a step of single tokens

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplusf_(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// conv channels: q (kv_heads * dim), then k (the same), then v (heads * vdim); taps_w [channels, taps] in that order
__global__ void __launch_bounds__(256)
delta_prepare_kernel(const float* __restrict__ proj, DeltaShape sh, const int32_t* __restrict__ token_seq,
                     const int32_t* __restrict__ q_start, const int32_t* __restrict__ state_slots,
                     const float* __restrict__ state, size_t state_stride, const float* __restrict__ taps_w,
                     const float* __restrict__ dt_pre, int ld_dt, const float* __restrict__ dt_bias,
                     const float* __restrict__ a_log, float* __restrict__ qn, float* __restrict__ kn,
                     float* __restrict__ vn, float* __restrict__ beta, float* __restrict__ decay,
                     float* __restrict__ kq) {
  extern __shared__ float act[];       // the token's channels after convolution and SiLU
  const int t = blockIdx.x;
  const int e = token_seq[t];
  const int n = t - q_start[e];        // the token's index inside its entry
  const int nqk = sh.kv_heads * sh.dim, nv = sh.heads * sh.vdim, channels = 2 * nqk + nv;
  if (blockIdx.y == 1) {
    // the token's second workgroup: the gates of the recurrence, which need nothing of the convolution
    for (int h = threadIdx.x; h < sh.heads; h += 256)
      beta[(size_t)t * sh.heads + h] = sigmoidf_(proj[(size_t)t * sh.ldp + sh.off_b + h]);
    const int nd = sh.heads * sh.dim;
    for (int c = threadIdx.x; c < nd; c += 256) {
      const float rate = expf(a_log[c / sh.dim]);
      decay[(size_t)t * nd + c] = expf(-rate * softplusf_(dt_pre[(size_t)t * ld_dt + c] + dt_bias[c]));
    }
    return;
  }
  const float* conv_state = state + (size_t)state_slots[e] * state_stride;
  // (unrolled so that the loads of several channels and taps are in flight together)
#pragma unroll 4
  for (int c = threadIdx.x; c < channels; c += 256) {
    const int col = c < nqk ? sh.off_q + c : c < 2 * nqk ? sh.off_k + (c - nqk) : sh.off_v + (c - 2 * nqk);
    float y = 0.f;
#pragma unroll 4
    for (int j = 0; j < sh.taps; ++j) {
      const int s = n - (sh.taps - 1) + j;      // index inside the entry of the input under tap j
      const float x = s >= 0 ? proj[(size_t)(t - (sh.taps - 1) + j) * sh.ldp + col]
                             : conv_state[(size_t)(sh.taps - 1 + s) * channels + c];
      y = fmaf(taps_w[(size_t)c * sh.taps + j], x, y);
    }
    act[c] = y * sigmoidf_(y);
  }
  __syncthreads();
  // unit length per head: a wave a head
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float q_scale = 1.0f / sqrtf((float)sh.dim);
  for (int hh = wave; hh < 2 * sh.kv_heads; hh += 4) {
    float* x = act + (size_t)hh * sh.dim;
    float ss = 0.f;
    for (int i = lane; i < sh.dim; i += 64) ss += x[i] * x[i];
    ss = wave_sum(ss);
    const bool is_q = hh < sh.kv_heads;
    const float inv = (is_q ? q_scale : 1.0f) / sqrtf(ss + 1e-6f);
    float* dst = (is_q ? qn : kn) + (size_t)t * nqk + (size_t)(is_q ? hh : hh - sh.kv_heads) * sh.dim;
    for (int i = lane; i < sh.dim; i += 64) dst[i] = act[(size_t)hh * sh.dim + i] = x[i] * inv;
  }
  __syncthreads();
  // k . q of every q/k head, which the recurrence's read-out needs once a token
  for (int hh = wave; hh < sh.kv_heads; hh += 4) {
    float d = 0.f;
    for (int i = lane; i < sh.dim; i += 64) d = fmaf(act[(size_t)hh * sh.dim + i], act[(size_t)(sh.kv_heads + hh) * sh.dim + i], d);
    d = wave_sum(d);
    if (lane == 0) kq[(size_t)t * sh.kv_heads + hh] = d;
  }
  for (int c = threadIdx.x; c < nv; c += 256) vn[(size_t)t * nv + c] = act[2 * nqk + c];
}

// one thread a (entry, channel): the state's rows in ascending order, so that a row is read before it is overwritten
__global__ void __launch_bounds__(256)
delta_conv_state_kernel(const float* __restrict__ proj, DeltaShape sh, const int32_t* __restrict__ q_start,
                        const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride) {
  const int e = blockIdx.y;
  const int nqk = sh.kv_heads * sh.dim, nv = sh.heads * sh.vdim, channels = 2 * nqk + nv;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= channels) return;
  const int first = q_start[e], count = q_start[e + 1] - first;
  const int col = c < nqk ? sh.off_q + c : c < 2 * nqk ? sh.off_k + (c - nqk) : sh.off_v + (c - 2 * nqk);
  float* st = state + (size_t)state_slots[e] * state_stride;
  const int keep = sh.taps - 1;
  for (int r = 0; r < keep; ++r) {
    const int s = count - keep + r;     // index inside the entry of the input that row r holds afterwards
    st[(size_t)r * channels + c] = s >= 0 ? proj[(size_t)(first + s) * sh.ldp + col] : st[(size_t)(r + count) * channels + c];
  }
}

// Sum over 32 or 16 neighbouring lanes; every lane gets the same sum (the pairs of each step add the same two numbers).
// x[0], x[1] of 16 lanes are what two neighbours of 32 have: the sums are the same bits.
__device__ __forceinline__ float row_sum(float x) {
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, false));    // lanes i ^ 1
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, false));    // lanes i ^ 2
  x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, false));   // the other quad of 8
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x140, 0xf, 0xf, false));   // the other half of 16
}
template <int LANES>
__device__ __forceinline__ float column_sum(const float (&x)[1]) {
  const float y = row_sum(x[0]);
  if constexpr (LANES == 16) return y;
  const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return __uint_as_float(rows[0]) + __uint_as_float(rows[1]);                                       // the other 16
}
template <int LANES>
__device__ __forceinline__ float column_sum(const float (&x)[2]) { return row_sum(x[0] + x[1]); }

// d1, d2: a column's sums of x1 and x2.  Where a column has two rows of 16 lanes, the swap that adds their neighbours (what a lane of 16
// adds by itself) leaves x1 in the first row and x2 in the second, so that the other four steps serve both.
template <int LANES, int G>
__device__ __forceinline__ void column_sums(const float (&x1)[G], const float (&x2)[G], float& d1, float& d2) {
  if constexpr (LANES == 32) {
    const auto half = __builtin_amdgcn_permlane16_swap(__float_as_uint(x1[0]), __float_as_uint(x2[0]), false, false);
    const uint32_t y = __float_as_uint(row_sum(__uint_as_float(half[0]) + __uint_as_float(half[1])));
    const auto both = __builtin_amdgcn_permlane16_swap(y, y, false, false);
    d1 = __uint_as_float(both[0]), d2 = __uint_as_float(both[1]);
  } else {
    d1 = column_sum<LANES>(x1), d2 = column_sum<LANES>(x2);
  }
}

// LANES (32 or 16) lanes share a column of S and hold G groups of R rows of it each, up to dim rows; a workgroup of four
// waves holds COLS columns.  The tokens' q, k, decay (for the head), v (for the columns), beta and k . q pass LDS in blocks
// of TB tokens: the next block is fetched from memory while this one is worked on, W values at a time (4 where dim allows it), and the
// next token's rows are read from LDS while this one's are worked on.
// Bound by a wave's instructions for a token, one after the other, and where the workgroups fill the CUs by all of them.  So a whole
// block is written out with every place in LDS a constant, and a lane keeps the output of one of its tokens for one store at the end: 36
// instructions a token with 32 lanes a column, where addresses, a branch and a store for each were as many as the arithmetic.
// us, before / now: one entry of 2,048 tokens, 8 heads of 128 x 128 433 / 248, of 64 x 64 339 / 206, of 256 x 128 593 / 407; 300
// tokens of 128 x 128 67 / 40, eight entries of 256 76 / 63; 8 and 64 single tokens beside each other 6.0 / 4.5 and 30.7 / 18.6 (their time
// is that of the state's way, four values a load where dim and the row allow it).
// 16 lanes a column need fewer instructions in all, 32 fewer in a row.  dim beyond 128 takes 32, whose rows would fill the registers
// otherwise; dim from 65 on takes 32 for entries long enough to leave CUs idle else (scan_wide); up to 64 rows 32 lanes give 2 percent to
// such entries and take up to 40 from others, so they take 16.  The sums are the same bits either way.

struct ScanArgs {
  const float *qn, *kn, *vn, *beta, *decay, *kq;
  DeltaShape sh;
  const int32_t *q_start, *state_slots;
  float* state;
  size_t state_stride, s_offset;
  float* o;
  int n_tokens, n_entries;
  int long_from;      // entries of so many tokens and more are begun before the others
};

// An entry's columns take 32 lanes each where as many workgroups as the step's tokens would make of such entries are about one a CU or fewer
// (a sixteenth more leaves an entry beside single tokens in).  us with 32 / 16 lanes, heads of 128 x 128: 8 heads, one entry of 2,048 (128
// workgroups) 249 / 300, the same beside 63 single tokens 242 / 294, two of 1,024 (256) 128 / 151; 16 heads, 2,041 tokens and seven single ones
// (257) 251 / 303.  Beyond: 12 heads, 1,400 and 640 tokens (280) 211 / 208; 16 heads, the same (373) 213 / 209; 8 heads, three of 682 (384)
// 107 / 103, four of 512 82 / 78.  (Some counts there leave 16 lanes the worse split, 12 heads, four of 512 107 / 119, but no rule tells them.)
constexpr int kScanGroups = 272;
__host__ __device__ __forceinline__ bool scan_wide(const DeltaShape& sh, int count, int n_tokens) {
  return (int64_t)sh.heads * ((sh.vdim + 7) / 8) * n_tokens <= (int64_t)kScanGroups * count;
}
template <int R, int G, int LANES>
struct ScanBlock {
  static constexpr int DP = LANES * G * R;            // dim rounded up; rows beyond dim hold zeros
  static constexpr int TB = R <= 4 ? 16 : 8;          // tokens a block
  static constexpr int COLS = 256 / LANES;
  static constexpr int FLOATS = 2 * TB * (3 * DP + COLS + 2);       // of LDS
};
#if defined(__HIP_DEVICE_COMPILE__)
// columns group * COLS and on of a head's state, for tokens first .. first + count - 1
template <int R, int G, int LANES, int W>
__device__ __forceinline__ void scan_columns(const ScanArgs& a, int group, int h, int e, int first, int count, float* __restrict__ lds) {
  using C = ScanBlock<R, G, LANES>;
  constexpr int DP = C::DP, TB = C::TB, COLS = C::COLS;
  constexpr int PER = (TB * DP / W + 255) / 256;       // pieces of W values of q (k, decay) a thread fetches a block
  constexpr int RW = W < R ? W : R;                    // rows of the state a load takes
  static_assert((LANES == 16 || G == 1) && R % RW == 0, "");
  typedef float piece_t __attribute__((ext_vector_type(W)));
  typedef float four_t __attribute__((ext_vector_type(4)));
  typedef float rows_t __attribute__((ext_vector_type(RW)));
  const DeltaShape& sh = a.sh;
  auto& sq = *reinterpret_cast<float(*)[2][TB][DP]>(lds);
  auto& sk = *reinterpret_cast<float(*)[2][TB][DP]>(lds + 2 * TB * DP);
  auto& sg = *reinterpret_cast<float(*)[2][TB][DP]>(lds + 4 * TB * DP);
  auto& sv = *reinterpret_cast<float(*)[2][COLS][TB]>(lds + 6 * TB * DP);
  auto& sb = *reinterpret_cast<float(*)[2][TB]>(lds + 6 * TB * DP + 2 * TB * COLS);
  auto& skq = *reinterpret_cast<float(*)[2][TB]>(lds + 6 * TB * DP + 2 * TB * COLS + 2 * TB);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int part = lane & (LANES - 1);
  const int col_local = wave * (64 / LANES) + lane / LANES;
  const int col = group * COLS + col_local;
  const int kv = h / (sh.heads / sh.kv_heads);
  const int dim = sh.dim, vdim = sh.vdim;
  const bool col_ok = col < vdim;
  const int i0 = (LANES == 32 ? (part & 15) * 2 + (part >> 4) : part) * G * R;      // (neighbouring groups in the two rows)
  float* sp = a.state + (size_t)a.state_slots[e] * a.state_stride + a.s_offset +
              ((size_t)h * vdim + (col_ok ? col : 0)) * dim + i0;
  float s[G * R];
#pragma unroll
  for (int r = 0; r < G * R; r += RW) {
    const rows_t x = col_ok && i0 + r < dim ? *reinterpret_cast<const rows_t*>(sp + r) : rows_t(0.f);
#pragma unroll
    for (int i = 0; i < RW; ++i) s[r + i] = x[i];
  }

  const int nqk = sh.kv_heads * dim, nd = sh.heads * dim, nv = sh.heads * vdim;
  // block b's share of this thread: piece idx = tid + j * 256 of [TB][DP / W]; v: thread tid of [TB][COLS]; beta, k . q: tid < TB.
  // (Loads stand under no condition, which the compiler would wait for where the branches meet: what lies beyond the entry's tokens, dim
  // or vdim is out of the buffer's range and comes as zero.)
  constexpr uint32_t kOutside = 0x80000000u;
  uint32_t to_qk[PER], to_g[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int idx = tid + j * 256, tok = idx / (DP / W), i = idx % (DP / W) * W;
    const bool there = idx < TB * DP / W && i < dim;
    to_qk[j] = there ? (uint32_t)(tok * nqk + i) * 4 : kOutside;
    to_g[j] = there ? (uint32_t)(tok * nd + i) * 4 : kOutside;
  }
  const int cols = min(COLS, vdim - group * COLS);
  const uint32_t to_v = tid < TB * COLS && tid % COLS < cols ? (uint32_t)(tid / COLS * nv + tid % COLS) * 4 : kOutside;
  const uint32_t to_b = tid < TB ? (uint32_t)(tid * sh.heads) * 4 : kOutside, to_kq = tid < TB ? (uint32_t)(tid * sh.kv_heads) * 4 : kOutside;
  piece_t pq[PER], pk[PER], pg[PER];
  float pv = 0.f, pb = 0.f, pkq = 0.f;
  auto fetch = [&](int b) {
    const size_t t = (size_t)(first + b * TB);
    const int rows = min(TB, count - b * TB);
    auto some = [&](const float* p, int ld, int width) {
      return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, ((rows - 1) * ld + width) * 4, 0x00027000);
    };
    const auto q_b = some(a.qn + t * nqk + (size_t)kv * dim, nqk, dim), k_b = some(a.kn + t * nqk + (size_t)kv * dim, nqk, dim);
    const auto g_b = some(a.decay + t * nd + (size_t)h * dim, nd, dim);
    auto piece = [&](auto from, uint32_t at) {
      if constexpr (W == 4) return __builtin_bit_cast(piece_t, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
      else return __builtin_bit_cast(piece_t, __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0));
    };
#pragma unroll
    for (int j = 0; j < PER; ++j) pq[j] = piece(q_b, to_qk[j]), pk[j] = piece(k_b, to_qk[j]), pg[j] = piece(g_b, to_g[j]);
    auto one = [&](auto from, uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0)); };
    pv = one(some(a.vn + t * nv + (size_t)h * vdim + (size_t)group * COLS, nv, cols), to_v);
    pb = one(some(a.beta + t * sh.heads + h, sh.heads, 1), to_b);
    pkq = one(some(a.kq + t * sh.kv_heads + kv, sh.kv_heads, 1), to_kq);
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int idx = tid + j * 256;
      if (TB * DP / W % 256 != 0 && idx >= TB * DP / W) continue;
      *reinterpret_cast<piece_t*>(&sq[buf][0][0] + idx * W) = pq[j];
      *reinterpret_cast<piece_t*>(&sk[buf][0][0] + idx * W) = pk[j];
      *reinterpret_cast<piece_t*>(&sg[buf][0][0] + idx * W) = pg[j];
    }
    if (tid < TB * COLS) sv[buf][tid % COLS][tid / COLS] = pv;
    if (tid < TB) sb[buf][tid] = pb, skq[buf][tid] = pkq;
  };
  struct Rows { float k[G * R], g[G * R], q[G * R]; };
  auto load = [&](Rows& x, int buf, int tok) {
#pragma unroll
    for (int r = 0; r < G * R; ++r) x.k[r] = sk[buf][tok][i0 + r], x.g[r] = sg[buf][tok][i0 + r], x.q[r] = sq[buf][tok][i0 + r];
  };
  float out = 0.f;       // of the block's token `part`
  auto token = [&](const Rows& x, float v, float b, float kq_, int tok) {
    float p1[G], p2[G];
#pragma unroll
    for (int g = 0; g < G; ++g) p1[g] = p2[g] = 0.f;
#pragma unroll
    for (int r = 0; r < G * R; ++r) {
      s[r] *= x.g[r];
      p1[r / R] = fmaf(s[r], x.k[r], p1[r / R]);
      p2[r / R] = fmaf(s[r], x.q[r], p2[r / R]);
    }
    float d1, d2;
    column_sums<LANES>(p1, p2, d1, d2);
    const float u = b * (v - d1);
    // o = S_new^T q with S_new = diag(g) S + k u^T
    out = part == tok ? fmaf(u, kq_, d2) : out;
#pragma unroll
    for (int r = 0; r < G * R; ++r) s[r] = fmaf(x.k[r], u, s[r]);
  };
  const int blocks = (count + TB - 1) / TB;
  if (blocks > 0) {
    fetch(0);
    stash(0);
  }
  // (the state has arrived, which the compiler would else make sure of in front of every block's tokens, by waiting for
  // everything, the next block's fetch with it)
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
  __syncthreads();
  for (int b = 0; b < blocks; ++b) {
    const int buf = b & 1;
    if (b + 1 < blocks) fetch(b + 1);
    const int n_tok = min(TB, count - b * TB);
    if (n_tok == TB) {
      // the rows are read two tokens before their turn, what every lane of a column needs by fours
      Rows x[3];
      four_t v[2], be[2], kq4[2];
      auto load_four = [&](int tok) {
        const int i = (tok >> 2) & 1;
        v[i] = *reinterpret_cast<const four_t*>(&sv[buf][col_local][tok]);
        be[i] = *reinterpret_cast<const four_t*>(&sb[buf][tok]);
        kq4[i] = *reinterpret_cast<const four_t*>(&skq[buf][tok]);
      };
      load(x[0], buf, 0);
      load_four(0);
      load(x[1], buf, 1);
#pragma unroll
      for (int tok = 0; tok < TB; ++tok) {
        __builtin_amdgcn_sched_barrier(0);       // (the compiler would read them when it needs them)
        if (tok + 2 < TB) load(x[(tok + 2) % 3], buf, tok + 2);
        if (tok % 4 == 2 && tok + 2 < TB) load_four(tok + 2);
        const int i = (tok >> 2) & 1, at = tok & 3;
        token(x[tok % 3], v[i][at], be[i][at], kq4[i][at], tok);
      }
    } else {
      Rows x, y;
      float v = sv[buf][col_local][0], be = sb[buf][0], kq1 = skq[buf][0];
      load(x, buf, 0);
#pragma unroll 1
      for (int tok = 0; tok < n_tok; ++tok) {
        load(y, buf, tok + 1);      // (there is one: n_tok < TB)
        const float next_v = sv[buf][col_local][tok + 1], next_b = sb[buf][tok + 1], next_kq = skq[buf][tok + 1];
        token(x, v, be, kq1, tok);
        x = y, v = next_v, be = next_b, kq1 = next_kq;
      }
    }
    if (part < n_tok && col_ok) a.o[(size_t)(first + b * TB + part) * nv + (size_t)h * vdim + col] = out;
    if (b + 1 < blocks) stash(buf ^ 1);
    __syncthreads();
  }
  if (col_ok) {
#pragma unroll
    for (int r = 0; r < G * R; r += RW) {
      rows_t x;
#pragma unroll
      for (int i = 0; i < RW; ++i) x[i] = s[r + i];
      if (i0 + r < dim) *reinterpret_cast<rows_t*>(sp + r) = x;
    }
  }
}
#endif

// A step's portions of prompts begin before its single tokens, wherever they lie among them (ORDERED): one that begins late has a CU for itself
// only by chance.  Up to 64 entries are put in order; of more, those that end in a portion are taken from the last on, as steps are that have no
// portion, those that begin with one from the first on, and up to 256 others are put in order.  us in the entries' order, by the kernel whose
// blocks were not written out / from the last on / now: 32 heads of 128 x 128, 2,041 tokens behind seven single ones 452 / 305 / 302, in front of
// them 442 / 490 / 303; 8 heads, 1,985 in front of 63 432 / 308 / 242, 700 among 200 196 / 128 / 93, in front of them 153 / 148 / 93.
// Steps without a long entry lose by it (16 entries of three tokens 7.3 -> 7.8): those that can have none of kScanLong tokens are not looked at.
constexpr int kScanOrdered = 256, kScanLong = 128;
#if defined(__HIP_DEVICE_COMPILE__)
struct ScanEntry { int e, first, count; };
// The zth entry, long ones first.  Every wave looks at all of them, 64 at a time in one trip to memory, which tells it the entry's first token
// as well.
template <int CHUNKS>
__device__ __forceinline__ ScanEntry entry_among(const ScanArgs& a, int z) {
  const int lane = threadIdx.x & 63;
  int first[CHUNKS], count[CHUNKS], n_long = 0, n_short = 0;
  unsigned long long longs[CHUNKS], shorts[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = min(c * 64 + lane, a.n_entries - 1);
    first[c] = a.q_start[i], count[c] = a.q_start[i + 1];
  }
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    count[c] -= first[c];
    const bool there = c * 64 + lane < a.n_entries;
    longs[c] = __ballot(there && count[c] >= a.long_from), shorts[c] = __ballot(there && count[c] < a.long_from);
    n_short += __popcll(longs[c]);      // (short ones come behind all long ones)
  }
  auto before = [&](unsigned long long m) { return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0)); };
  ScanEntry found{0, 0, 0};
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const bool is_long = count[c] >= a.long_from;
    const int place = is_long ? n_long + before(longs[c]) : n_short + before(shorts[c]);
    const unsigned long long hit = __ballot(c * 64 + lane < a.n_entries && place == z);
    if (hit != 0) {
      const int at = __builtin_ctzll(hit);
      found = ScanEntry{c * 64 + at, __builtin_amdgcn_readlane(first[c], at), __builtin_amdgcn_readlane(count[c], at)};
    }
    n_long += __popcll(longs[c]), n_short += __popcll(shorts[c]);
  }
  return found;
}
template <bool ORDERED>
__device__ __forceinline__ ScanEntry entry_at(const ScanArgs& a, int z) {
  const int n = a.n_entries, e = n - 1 - z, first = a.q_start[e], end = a.q_start[e + 1];
  if constexpr (ORDERED) {
    if (n <= 64) return entry_among<1>(a, z);
    const int z_first = a.q_start[z], z_end = a.q_start[z + 1];
    if (a.q_start[n] - a.q_start[n - 1] < a.long_from) {
      if (a.q_start[1] - a.q_start[0] >= a.long_from) return ScanEntry{z, z_first, z_end - z_first};
      if (n <= kScanOrdered) return entry_among<kScanOrdered / 64>(a, z);
    }
  }
  return ScanEntry{e, first, end - first};
}
#endif

template <int R, int G, int LANES, int W, bool ORDERED>
__global__ void __launch_bounds__(256) delta_scan_kernel(ScanArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) float lds[ScanBlock<R, G, LANES>::FLOATS];
  const ScanEntry at = entry_at<ORDERED>(a, blockIdx.z);
  scan_columns<R, G, LANES, W>(a, blockIdx.x, blockIdx.y, at.e, at.first, at.count, lds);
#endif
}
// 32 lanes a column for the entries that have most of the step's tokens, 16 for the others.  The first `extra` of blockIdx.z count the
// former's, for the columns that 16 lanes would leave no workgroup; then all entries follow.
// (With workgroups without work between those with it, every second CU stayed idle: four entries of 512 tokens 118 us against 78.)
template <int R, int W, bool ORDERED>
__global__ void __launch_bounds__(256) delta_scan_long_kernel(ScanArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(16))) float lds[ScanBlock<R, 2, 16>::FLOATS];
  const int extra = (int)gridDim.z - a.n_entries;
  const bool more = (int)blockIdx.z < extra;
  ScanEntry at{-1, 0, 0};
  if (more) {
    int nth = blockIdx.z;
    for (int from = 0; from < a.n_entries; from += 64) {
      const int i = min(from + (int)(threadIdx.x & 63), a.n_entries - 1), first = a.q_start[i], count = a.q_start[i + 1] - first;
      unsigned long long wide = __ballot(from + (int)(threadIdx.x & 63) < a.n_entries && scan_wide(a.sh, count, a.n_tokens));
      for (; wide != 0 && nth > 0; --nth) wide &= wide - 1;
      if (wide != 0) {
        const int w = __builtin_ctzll(wide);
        at = ScanEntry{from + w, __builtin_amdgcn_readlane(first, w), __builtin_amdgcn_readlane(count, w)};
        break;
      }
    }
    if (at.e < 0) return;
  } else {
    at = entry_at<ORDERED>(a, (int)blockIdx.z - extra);
  }
  const int group = blockIdx.x + (more ? gridDim.x : 0);
  if (scan_wide(a.sh, at.count, a.n_tokens)) {
    if (group * 8 < a.sh.vdim) scan_columns<R, 1, 32, W>(a, group, blockIdx.y, at.e, at.first, at.count, lds);
  } else {
    scan_columns<R, 2, 16, W>(a, group, blockIdx.y, at.e, at.first, at.count, lds);
  }
#endif
}

template <typename TO>
__global__ void __launch_bounds__(256)
delta_out_kernel(const float* __restrict__ o, const float* __restrict__ gate_pre, int ld_gate,
                 const float* __restrict__ w, float eps, TO* __restrict__ out, int heads, int vdim) {
  const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int h = wave; h < heads; h += 4) {
    const size_t base = ((size_t)t * heads + h) * vdim;
    float ss = 0.f;
    for (int j = lane; j < vdim; j += 64) ss += o[base + j] * o[base + j];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)vdim + eps);
    for (int j = lane; j < vdim; j += 64)
      out[base + j] = from_f32<TO>(o[base + j] * inv * w[j] *
                                   sigmoidf_(gate_pre[(size_t)t * ld_gate + (size_t)h * vdim + j]));
  }
}

// A step of single tokens (every entry has one): all of the above in one launch, a workgroup a (q/k head, entry) with the heads that
// read that q/k head, so that what the convolution reads and replaces of the request's state belongs to one workgroup.  The state's
// columns, `PASSES` a thread at a time, are asked for before anything else and arrive while convolution, unit lengths and decays are
// made; the heads' outputs are normed from LDS.  Every sum is added in the order of the kernels above: the same bits.
// Bound by its trips to memory (the slot, then the state) and by what a CU moves of the state, 256 KB for two heads of 128 x 128: with
// eight requests of 8 heads over 4 q/k heads 32 workgroups, 12.6 us for the launch, where the four took 29.5 (prepare 11.7, the
// convolution's state 5.1, scan 8.2, since then 1.5 less, output 5.2).  (With the loads of the state, the taps and the gates each waited for
// by itself: 15.8.)
// A CU has one such workgroup at a time (heads of 64 and 128 take all 128 registers a thread may have, and three values spill around
// the passes), so steps of many small heads keep the four launches: delta_step_pays in ops.py.
template <int R, int G, int LANES, typename TO>
__global__ void __launch_bounds__(kStepThreads)
delta_step_kernel(const float* __restrict__ proj, DeltaShape sh, const int32_t* __restrict__ q_start,
                  const int32_t* __restrict__ state_slots, float* __restrict__ state, size_t state_stride, size_t s_offset,
                  const float* __restrict__ taps_w, const float* __restrict__ dt_pre, int ld_dt, const float* __restrict__ dt_bias,
                  const float* __restrict__ a_log, const float* __restrict__ gate_pre, int ld_gate,
                  const float* __restrict__ norm_w, float eps, TO* __restrict__ out, bool vec) {
  constexpr int GR = G * R, DP = LANES * GR, COLS = kStepThreads / LANES, PASSES = 32 / GR < 8 ? 32 / GR : 8;
  typedef float rows_t __attribute__((ext_vector_type(R)));
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kv = blockIdx.x, e = blockIdx.y;
  const int dim = sh.dim, vdim = sh.vdim, group = sh.heads / sh.kv_heads, h0 = kv * group, cols = group * vdim;
  const int nqk = sh.kv_heads * dim, nv = sh.heads * vdim, channels = 2 * nqk + nv, keep = sh.taps - 1;
  float* const q = lds;                      // [DP], zeros from dim on
  float* const k = q + DP;                   // [DP]
  float* const g = k + DP;                   // [group][DP]
  float* const v = g + group * DP;           // [cols]
  float* const o = v + cols;                 // [cols]
  float* const gate = o + cols;              // [cols]
  int* const head = reinterpret_cast<int*>(gate + cols);      // [cols] a column's head
  float* const beta = gate + 2 * cols;       // [group]
  const int t = q_start[e];
  float* const st = state + (size_t)state_slots[e] * state_stride;
  float* const sp = st + s_offset + (size_t)h0 * vdim * dim;      // column f of the workgroup's: at f * dim
  const int part = lane & (LANES - 1), i0 = part * GR, mine = tid / LANES;
  float s[PASSES][GR];
  auto load = [&](int f0) {
    if (vec) {
#pragma unroll
      for (int p = 0; p < PASSES; ++p)
#pragma unroll
        for (int j = 0; j < G; ++j) {
          const uint32_t at = (uint32_t)(min(f0 + p * COLS + mine, cols - 1) * dim + min(i0 + j * R, dim - R));
          const rows_t x = *reinterpret_cast<const rows_t*>(sp + at);
#pragma unroll
          for (int r = 0; r < R; ++r) s[p][j * R + r] = x[r];
        }
    } else {
#pragma unroll
      for (int p = 0; p < PASSES; ++p)
#pragma unroll
        for (int r = 0; r < GR; ++r) s[p][r] = sp[(uint32_t)(min(f0 + p * COLS + mine, cols - 1) * dim + min(i0 + r, dim - 1))];
    }
  };
  auto store = [&](int f0) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int f = f0 + p * COLS + mine;
      if (f >= cols) continue;
      const uint32_t to = (uint32_t)(f * dim + i0);
      if (vec) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
          rows_t x;
#pragma unroll
          for (int r = 0; r < R; ++r) x[r] = s[p][j * R + r];
          if (i0 + j * R < dim) *reinterpret_cast<rows_t*>(sp + (to + j * R)) = x;
        }
      } else {
#pragma unroll
        for (int r = 0; r < GR; ++r)
          if (i0 + r < dim) sp[to + r] = s[p][r];
      }
    }
  };
  load(0);
  // the workgroup's channels: q, k, then v
  const int own = 2 * dim + cols;
  auto channel = [&](int i) { return i < dim ? kv * dim + i : i < 2 * dim ? nqk + kv * dim + i - dim : 2 * nqk + h0 * vdim + i - 2 * dim; };
  auto input = [&](int i) {
    return proj[(size_t)t * sh.ldp + (i < dim ? sh.off_q + kv * dim + i : i < 2 * dim ? sh.off_k + kv * dim + i - dim
                                                                                     : sh.off_v + h0 * vdim + i - 2 * dim)];
  };
  float held[4], held_in = 0.f;              // of the thread's first channel: its earlier inputs and the token's
  // (channels, decays and gates are different threads' where there are enough: each is a trip to memory of its own)
  const int decays = own + group * DP, items = decays + cols;
  for (int i = tid; i < items; i += kStepThreads) {
    if (i < own) {
      const int c = channel(i);
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      const float in = input(i), y = convolve_one(st + c, taps_w + (size_t)c * sh.taps, keep, channels, in, 0.f, x);
      if (i == tid) {
        held_in = in;
#pragma unroll
        for (int j = 0; j < 4; ++j) held[j] = x[j];
      }
      (i < dim ? q + i : i < 2 * dim ? k + i - dim : v + i - 2 * dim)[0] = y * sigmoidf_(y);
    } else if (i < decays) {
      const int hl = (i - own) / DP, h = h0 + hl, d = min((i - own) % DP, dim - 1);
      const float pre = dt_pre[(size_t)t * ld_dt + (size_t)h * dim + d], bias = dt_bias[(size_t)h * dim + d], rate = expf(a_log[h]);
      g[i - own] = expf(-rate * softplusf_(pre + bias));      // (beyond dim: never used)
    } else {
      const int f = i - decays, hl = f / vdim;
      const float raw = gate_pre[(size_t)t * ld_gate + (size_t)h0 * vdim + f], b = proj[(size_t)t * sh.ldp + sh.off_b + h0 + hl];
      gate[f] = sigmoidf_(raw);
      head[f] = hl;
      beta[hl] = sigmoidf_(b);                                // (the same by all of the head's columns)
    }
  }
  for (int i = dim + tid; i < DP; i += kStepThreads) q[i] = k[i] = 0.f;
  lds_barrier();
  if (wave < 2) {
    float* const x = wave == 0 ? q : k;
    float ss = 0.f;
    for (int i = lane; i < dim; i += 64) ss += x[i] * x[i];
    ss = wave_sum(ss);
    const float inv = (wave == 0 ? 1.0f / sqrtf((float)dim) : 1.0f) / sqrtf(ss + 1e-6f);
    for (int i = lane; i < dim; i += 64) x[i] = x[i] * inv;
  }
  lds_barrier();
  float kq = 0.f;                            // k . q
  for (int i = lane; i < dim; i += 64) kq = fmaf(q[i], k[i], kq);
  kq = wave_sum(kq);
  float kr[GR], qr[GR];
#pragma unroll
  for (int r = 0; r < GR; ++r) kr[r] = k[i0 + r], qr[r] = q[i0 + r];
  for (int f0 = 0; f0 < cols; f0 += PASSES * COLS) {
    if (f0 > 0) load(f0);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int f = f0 + p * COLS + mine, there = min(f, cols - 1), hl = head[there];
      float p1[G], p2[G];
#pragma unroll
      for (int j = 0; j < G; ++j) p1[j] = p2[j] = 0.f;
#pragma unroll
      for (int r = 0; r < GR; ++r) {
        // (what was fetched for a row beyond dim is another row's; made zero here and not at the load, which would then stand
        // under the condition and be waited for at once)
        s[p][r] = i0 + r < dim ? s[p][r] * g[hl * DP + i0 + r] : 0.f;
        p1[r / R] = fmaf(s[p][r], kr[r], p1[r / R]);
        p2[r / R] = fmaf(s[p][r], qr[r], p2[r / R]);
      }
      const float d1 = column_sum<LANES>(p1), d2 = column_sum<LANES>(p2);
      const float u = beta[hl] * (v[there] - d1);
      if (part == 0 && f < cols) o[f] = fmaf(u, kq, d2);
#pragma unroll
      for (int r = 0; r < GR; ++r) s[p][r] = fmaf(kr[r], u, s[p][r]);
    }
    store(f0);
  }
  for (int i = tid; i < own; i += kStepThreads) push_inputs(st + channel(i), keep, channels, i == tid ? held_in : input(i), held, i == tid);
  lds_barrier();
  for (int hl = wave; hl < group; hl += kStepThreads / kWave) {
    const float* const oh = o + hl * vdim;
    float ss = 0.f;
    for (int j = lane; j < vdim; j += 64) ss += oh[j] * oh[j];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)vdim + eps);
    for (int j = lane; j < vdim; j += 64)
      out[((size_t)t * sh.heads + h0 + hl) * vdim + j] = from_f32<TO>(oh[j] * inv * norm_w[j] * gate[hl * vdim + j]);
  }
}

// The second half of a low-rank map for few tokens: out[t, n] = sum_k x[t, k] * w[n, k], K small (the inner size of
// the map).  A thread an output; the token's K inputs wait in LDS.  With many tokens the general product is the better
// kernel (it reads a tile of w once for 64 tokens); the sums are added in its order (gemm_f32_tile.h), so that a token's
// are the same by both.
template <typename TW>
__global__ void __launch_bounds__(256)
lowrank_up_kernel(const float* __restrict__ x, int ldx, const TW* __restrict__ w, float* __restrict__ out, int ldo,
                  int N, int K) {
  extern __shared__ float xs[];
  const int t = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x;
  for (int k = threadIdx.x; k < (K + kF32Step - 1) / kF32Step * kF32Step; k += 256) xs[k] = k < K ? x[(size_t)t * ldx + k] : 0.f;
  __syncthreads();
  if (n >= N) return;
  const TW* wr = w + (size_t)n * K;
  const int steps = (K + kF32Step - 1) / kF32Step, whole = K / kF32Step, bits = f32_part_bits(N);
  float total = 0.f;
  for (int part = 0; part < 1 << bits; ++part) {
    const int end = f32_part_begin(steps, part + 1, bits);
    float acc = 0.f;
    for (int s = f32_part_begin(steps, part, bits); s < end; ++s) {
      const int k0 = s * kF32Step;
      float wv[kF32Step];
      if (s < whole) {
#pragma unroll
        for (int i = 0; i < kF32Step; ++i) wv[i] = to_f32(wr[k0 + i]);
      } else {
#pragma unroll
        for (int i = 0; i < kF32Step; ++i) wv[i] = k0 + i < K ? to_f32(wr[k0 + i]) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc = fmaf(xs[k0 + 8 * g + j], wv[8 * g + j], acc);
    }
    total += acc;
  }
  out[(size_t)t * ldo + n] = total;
}

// The same against a bfloat16 weight, on the matrix cores as the general product does it: a wave takes sixteen tokens against
// sixteen rows of the weight.
template <bool VEC>
__global__ void __launch_bounds__(256)
lowrank_split_kernel(const float* __restrict__ x, const bf16_t* __restrict__ w, float* __restrict__ out, int T, int N, int K, int ldx,
                     int ldo) {
  const int lane = threadIdx.x & 63, r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 64 + (threadIdx.x >> 6) * 16, t = blockIdx.y * 16 + r16;
  if (n0 >= N) return;
  const float* const xr = x + (size_t)min(t, T - 1) * ldx;             // (rows past the end: the last, never stored)
  const bf16_t* const wr = w + (size_t)min(n0 + r16, N - 1) * K;
  const int steps = (K + kF32Step - 1) / kF32Step, bits = f32_part_bits(N);
  f32x4_t total = {0.f, 0.f, 0.f, 0.f}, acc = total;
  int part = 0, next = f32_part_begin(steps, 1, bits);
  for (int s = 0; s < steps; ++s) {
    if (s == next) {
      total += acc;
      acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
      do next = f32_part_begin(steps, ++part + 1, bits);
      while (next == s);
    }
    f32x4_t xv[2];
    uint4 wv;
    split_load<VEC>(xr, s * kF32Step + kg * 8, K, xv);
    split_load<VEC>(wr, s * kF32Step + kg * 8, K, wv);
    const Split8 p = split_of(xv);
    const bf16x8_t whole = __builtin_bit_cast(bf16x8_t, wv), finite = split_weight(whole);
#pragma unroll
    for (int q = 0; q < 3; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q == 0 ? whole : finite, p.p[q], acc, 0, 0, 0);
  }
  total += acc;
  if (t >= T) return;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n0 + kg * 4 + e < N) out[(size_t)t * ldo + n0 + kg * 4 + e] = total[e];
}

extern "C" int atoma_lowrank_up(const float* x, int ldx, const void* w, int w_dtype, float* out, int ldo, int n_tokens,
                                int N, int K, hipStream_t stream) {
  if (n_tokens <= 0 || N <= 0) return 0;
  if (K <= 0 || K > 8192 || ldx < K || ldo < N || n_tokens > 65535) return ATOMA_ERR_SHAPE;
  const size_t lds = (size_t)(K + kF32Step - 1) / kF32Step * kF32Step * sizeof(float);
  dim3 grid((N + 255) / 256, n_tokens), block(256);
  if (w_dtype == kBF16 && split_product(N, K)) {
    const bool vec = K % kF32Step == 0 && ldx % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0;
    grid = dim3((N + 63) / 64, (n_tokens + 15) / 16);
    if (vec) hipLaunchKernelGGL((lowrank_split_kernel<true>), grid, block, 0, stream, x, (const bf16_t*)w, out, n_tokens, N, K, ldx, ldo);
    else hipLaunchKernelGGL((lowrank_split_kernel<false>), grid, block, 0, stream, x, (const bf16_t*)w, out, n_tokens, N, K, ldx, ldo);
  } else if (w_dtype == kBF16)
    hipLaunchKernelGGL((lowrank_up_kernel<bf16_t>), grid, block, lds, stream, x, ldx, (const bf16_t*)w, out, ldo, N, K);
  else if (w_dtype == kF32)
    hipLaunchKernelGGL((lowrank_up_kernel<float>), grid, block, lds, stream, x, ldx, (const float*)w, out,
                       ldo, N, K);
  else
    return ATOMA_ERR_DTYPE;
  ATOMA_LAUNCH_CHECK();
  return 0;
}

static bool shape_ok(const DeltaShape& sh) {
  return sh.heads > 0 && sh.kv_heads > 0 && sh.heads % sh.kv_heads == 0 && sh.dim > 0 && sh.dim <= 256 && sh.vdim > 0 &&
         sh.taps >= 1 && sh.taps <= 64 && sh.ldp > 0;
}

// Whether a token's q, k and v channels fit the LDS that delta_prepare keeps them in
static bool channels_fit(const DeltaShape& sh) {
  return (2 * (size_t)sh.kv_heads * sh.dim + (size_t)sh.heads * sh.vdim) * sizeof(float) <= 60 * 1024;
}

extern "C" int atoma_delta_prepare(const float* proj, int ldp, int off_q, int off_k, int off_v, int off_b, int heads,
                                   int kv_heads, int dim, int vdim, int taps, const int32_t* token_seq,
                                   const int32_t* q_start, const int32_t* state_slots, float* state,
                                   size_t state_stride, const float* taps_w, const float* dt_pre, int ld_dt,
                                   const float* dt_bias,
                                   const float* a_log, float* qn, float* kn, float* vn, float* beta, float* decay,
                                   float* kq, int n_tokens, int n_entries, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  DeltaShape sh{heads, kv_heads, dim, vdim, taps, ldp, off_q, off_k, off_v, off_b};
  if (!shape_ok(sh) || n_entries <= 0 || n_entries > 65535) return ATOMA_ERR_SHAPE;
  // (a token has two workgroups: convolution, SiLU and unit lengths; beta and decay)
  const int channels = 2 * kv_heads * dim + heads * vdim;
  if (!channels_fit(sh)) return ATOMA_ERR_SHAPE;
  hipLaunchKernelGGL(delta_prepare_kernel, dim3(n_tokens, 2), dim3(256), channels * sizeof(float), stream, proj, sh,
                     token_seq, q_start, state_slots, state, state_stride, taps_w, dt_pre, ld_dt, dt_bias, a_log, qn, kn, vn,
                     beta, decay, kq);
  ATOMA_LAUNCH_CHECK();
  if (taps > 1) {
    hipLaunchKernelGGL(delta_conv_state_kernel, dim3((channels + 255) / 256, n_entries), dim3(256), 0, stream, proj, sh,
                       q_start, state_slots, state, state_stride);
    ATOMA_LAUNCH_CHECK();
  }
  return 0;
}

extern "C" int atoma_delta_scan(const float* qn, const float* kn, const float* vn, const float* beta,
                                const float* decay, const float* kq, int heads, int kv_heads, int dim, int vdim, int taps,
                                const int32_t* q_start, const int32_t* state_slots, float* state, size_t state_stride,
                                int n_entries, int n_tokens, float* o, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  DeltaShape sh{heads, kv_heads, dim, vdim, taps, 1, 0, 0, 0, 0};
  if (!shape_ok(sh) || n_entries > 65535 || heads > 65535) return ATOMA_ERR_SHAPE;
  const size_t s_offset = (size_t)(taps - 1) * (2 * kv_heads * dim + heads * vdim);
  // (the longest entry there can be)
  const bool mixed = dim > 64 && dim <= 128 && n_entries < 32768 && scan_wide(sh, n_tokens - n_entries + 1, n_tokens);
  const int cols = dim > 128 ? 8 : 16;
  // (as many entries can have 32 lanes a column at most)
  const int extra = mixed ? std::min(n_entries, kScanGroups / (heads * ((vdim + 7) / 8))) : 0;
  const dim3 grid((vdim + cols - 1) / cols, heads, n_entries + extra), block(256);
  const bool four = dim % 4 == 0 && s_offset % 4 == 0 && state_stride % 4 == 0 &&
                    ((uintptr_t)qn | (uintptr_t)kn | (uintptr_t)decay | (uintptr_t)state) % 16 == 0;
  const bool ordered = n_entries > 1 && n_tokens - n_entries + 1 >= kScanLong;
  const int long_from = (int)std::min<int64_t>((int64_t)2 * n_tokens / n_entries + 1, n_tokens);      // (more than twice the mean)
  const ScanArgs args{qn, kn, vn, beta, decay, kq, sh, q_start, state_slots, state, state_stride, s_offset, o, n_tokens, n_entries, long_from};
#define ATOMA_SCAN(KERNEL, ...)                                                                                           \
  do {                                                                                                                    \
    if (four && ordered) hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 4, true>), grid, block, 0, stream, args);                \
    else if (four) hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 4, false>), grid, block, 0, stream, args);                     \
    else if (ordered) hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 1, true>), grid, block, 0, stream, args);                   \
    else hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 1, false>), grid, block, 0, stream, args);                               \
  } while (0)
  if (dim <= 16) ATOMA_SCAN(delta_scan_kernel, 1, 1, 16);
  else if (dim <= 32) ATOMA_SCAN(delta_scan_kernel, 1, 2, 16);
  else if (dim <= 64) ATOMA_SCAN(delta_scan_kernel, 2, 2, 16);
  else if (mixed) ATOMA_SCAN(delta_scan_long_kernel, 4);
  else if (dim <= 128) ATOMA_SCAN(delta_scan_kernel, 4, 2, 16);
  else ATOMA_SCAN(delta_scan_kernel, 8, 1, 32);
#undef ATOMA_SCAN
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_delta_out(const float* o, const float* gate_pre, int ld_gate, const float* w, float eps, void* out,
                               int out_dtype, int n_tokens, int heads, int vdim, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (heads <= 0 || vdim <= 0 || ld_gate < heads * vdim) return ATOMA_ERR_SHAPE;
  if (out_dtype == kF32)
    hipLaunchKernelGGL((delta_out_kernel<float>), dim3(n_tokens), dim3(256), 0, stream, o, gate_pre, ld_gate, w,
                       eps, (float*)out, heads, vdim);
  else if (out_dtype == kBF16)
    hipLaunchKernelGGL((delta_out_kernel<bf16_t>), dim3(n_tokens), dim3(256), 0, stream, o, gate_pre, ld_gate, w,
                       eps, (bf16_t*)out, heads, vdim);
  else
    return ATOMA_ERR_DTYPE;
  ATOMA_LAUNCH_CHECK();
  return 0;
}

static size_t step_lds_floats(const DeltaShape& sh, int dp) {
  const size_t group = sh.heads / sh.kv_heads, cols = group * sh.vdim;
  return 2 * dp + group * dp + 4 * cols + group;
}
static int padded_dim(int dim) { return dim <= 16 ? 16 : dim <= 32 ? 32 : dim <= 64 ? 64 : dim <= 128 ? 128 : 256; }

// Whether delta_step_kernel takes heads of these sizes: its vectors fit LDS, and a workgroup's state is at most 256 KB, beyond which the
// scan's many workgroups are the better split (at 256 KB, four heads of 128 x 128 to a q/k head, one request takes 14.9 us here and 16.3
// by the four launches, 64 requests 27.6 and 54.5).
// It takes none that atoma_delta_prepare refuses, whose rows of channels wait in LDS: a layer's prompts and its decoded tokens are
// refused alike.
extern "C" int atoma_delta_step_fits(int heads, int kv_heads, int dim, int vdim, int taps) {
  const DeltaShape sh{heads, kv_heads, dim, vdim, taps, 1, 0, 0, 0, 0};
  return shape_ok(sh) && kv_heads <= 65535 && channels_fit(sh) && (size_t)(heads / kv_heads) * vdim * dim <= 65536 &&
         step_lds_floats(sh, padded_dim(dim)) * sizeof(float) <= 60 * 1024;
}

// One token of every entry: what atoma_delta_prepare, atoma_delta_scan and atoma_delta_out do in turn.
extern "C" int atoma_delta_step(const float* proj, int ldp, int off_q, int off_k, int off_v, int off_b, int heads, int kv_heads,
                                int dim, int vdim, int taps, const int32_t* q_start, const int32_t* state_slots, float* state,
                                size_t state_stride, const float* taps_w, const float* dt_pre, int ld_dt, const float* dt_bias,
                                const float* a_log, const float* gate_pre, int ld_gate, const float* norm_w, float eps, void* out,
                                int out_dtype, int n_entries, hipStream_t stream) {
  if (n_entries <= 0) return 0;
  const DeltaShape sh{heads, kv_heads, dim, vdim, taps, ldp, off_q, off_k, off_v, off_b};
  if (!shape_ok(sh) || !atoma_delta_step_fits(heads, kv_heads, dim, vdim, taps) || n_entries > 65535) return ATOMA_ERR_SHAPE;
  const size_t s_offset = (size_t)(taps - 1) * (2 * kv_heads * dim + heads * vdim);
  const size_t lds = step_lds_floats(sh, padded_dim(dim)) * sizeof(float);
  const bool vec = dim % 8 == 0 && s_offset % 8 == 0 && state_stride % 8 == 0 && (uintptr_t)state % 32 == 0;
  const dim3 grid(kv_heads, n_entries), block(kStepThreads);
#define ATOMA_STEP(R, G, LANES, TO)                                                                                              \
  hipLaunchKernelGGL((delta_step_kernel<R, G, LANES, TO>), grid, block, lds, stream, proj, sh, q_start, state_slots, state,       \
                     state_stride, s_offset, taps_w, dt_pre, ld_dt, dt_bias, a_log, gate_pre, ld_gate, norm_w, eps, (TO*)out, vec)
#define ATOMA_STEP_BY_DIM(TO)                        \
  do {                                               \
    if (dim <= 16) ATOMA_STEP(1, 1, 16, TO);         \
    else if (dim <= 32) ATOMA_STEP(1, 2, 16, TO);    \
    else if (dim <= 64) ATOMA_STEP(2, 2, 16, TO);    \
    else if (dim <= 128) ATOMA_STEP(4, 1, 32, TO);   \
    else ATOMA_STEP(8, 1, 32, TO);                   \
  } while (0)
  if (out_dtype == kF32) ATOMA_STEP_BY_DIM(float);
  else if (out_dtype == kBF16) ATOMA_STEP_BY_DIM(bf16_t);
  else return ATOMA_ERR_DTYPE;
#undef ATOMA_STEP_BY_DIM
#undef ATOMA_STEP
  ATOMA_LAUNCH_CHECK();
  return 0;
}
