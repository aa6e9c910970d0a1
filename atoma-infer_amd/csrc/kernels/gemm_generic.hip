// C[M, N] = A[M, K] * W[N, K]^T in true float32: products and sums are float32 fused multiply-adds (on the matrix
// cores' float32 instruction), no reduced-precision mode.  A and W may be float32 or bfloat16 (widened exactly on
// load); C float32 or bfloat16.  Any M, N, K.  It is the product of the 32-bit path and the fallback for shapes the
// bfloat16 kernels refuse.
//
// Weights are [out, in] row-major as checkpoints store them (models/src/llama.rs:322-325), so both operands
// are contiguous along K.  Two kernels:
//
//   f32_tile_kernel    tiles of 128 x 128 (64 x 64 where those would leave CUs idle) through LDS, see gemm_f32_tile.h.
//                      Bound by the matrix cores (a float32 MFMA has a sixteenth of the bfloat16 rate);
//   f32_stream_kernel  up to 64 rows of A a workgroup against 16 rows of W, which come straight from memory, once: K is
//                      split over the workgroup's waves, whose sums meet in LDS.  Bound by W's bytes up to 16 rows of A.
//                      It also takes more rows where tiles of 64 x 64 would be fewer than the CUs (four waves of a tile
//                      walk all of K, eight of a streaming workgroup an eighth of it each).
//
// Measured on MI355X, float32 rows against bfloat16 weights, beside the one kernel of vector multiply-adds before (a tile
// of 64 x 64 a workgroup, 4 x 4 outputs a thread): the four layers of Llama 1B sizes and its head, 836 rows in one step
// and 16 steps of 4 rows, 106.5 -> 9.8 ms in all; gate-up (16,384 x 2,048) with 836 rows 622 us (90 TFLOP/s, 727 with
// loads under conditions; the card's float32 product of 8,192^3 reaches 153), with 4 rows 17.5 us (22.7 with one batch of
// loads in flight); the head (128,256 x 2,048) with 4 rows 117 us (133).
//
// The order in which an output's K products are summed depends on the kernel and on (N, K), not on its row's place.
#include "gemm_f32_tile.h"

using namespace atoma;

template <int T, bool VEC, typename TA, typename TW, typename TC>
__global__ void __launch_bounds__(256)
f32_tile_kernel(const TA* __restrict__ a, const TW* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                int ldw, int ldc) {
  __shared__ __attribute__((aligned(16))) float lds[2 * 2 * T * kF32Row];
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  f32x4_t acc[T / 32][T / 32];
#pragma unroll
  for (int i = 0; i < T / 32; ++i)
#pragma unroll
    for (int j = 0; j < T / 32; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32_tile<T, T, VEC, TA, TW>(
      lds, K, [&](int r) { return a + (size_t)min(m0 + r, M - 1) * lda; },
      [&](int r) { return w + (size_t)min(n0 + r, N - 1) * ldw; }, [](int) { return 1.f; }, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < T / 32; ++j) {
    const int m = m0 + (wave >> 1) * (T / 2) + j * 16 + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < T / 32; ++i) {
      const int n = n0 + (wave & 1) * (T / 2) + i * 16 + (lane >> 4) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) c[(size_t)m * ldc + n + e] = from_f32<TC>(acc[i][j][e]);
    }
  }
}

// eight neighbouring values of a row as they come from memory (16-byte aligned), and one of them as float32
template <typename T> struct Eight { f32x4_t lo, hi; };
template <> struct Eight<bf16_t> { uint4 v; };
__device__ __forceinline__ void fetch8(const float* p, Eight<float>& x) {
  x.lo = *reinterpret_cast<const f32x4_t*>(p), x.hi = *reinterpret_cast<const f32x4_t*>(p + 4);
}
__device__ __forceinline__ void fetch8(const bf16_t* p, Eight<bf16_t>& x) { x.v = *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ float value8(const Eight<float>& x, int e) { return e < 4 ? x.lo[e & 3] : x.hi[e & 3]; }
__device__ __forceinline__ float value8(const Eight<bf16_t>& x, int e) {
  const uint32_t q = e < 2 ? x.v.x : e < 4 ? x.v.y : e < 6 ? x.v.z : x.v.w;
  return __uint_as_float(e & 1 ? q & 0xffff0000u : q << 16);
}

// MT blocks of 16 rows of A; WK waves that split K (K % 32 == 0; rows of A and W aligned to 16 bytes).  A step is 32
// values of K: lane group g holds values 8 g .. 8 g + 7, and MFMA j sums the values 8 g + j.
template <int MT, int WK, typename TA, typename TW, typename TC>
__global__ void __launch_bounds__(64 * WK)
f32_stream_kernel(const TA* __restrict__ a, const TW* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                  int ldw, int ldc) {
  constexpr int U = MT == 1 ? 4 : 2;       // steps whose loads are in flight together
  __shared__ f32x4_t red[WK - 1][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
  const int steps = K / 32, begin = steps * wave / WK, end = steps * (wave + 1) / WK;
  const TW* const wp = w + (size_t)min(n0 + r16, N - 1) * ldw + kg * 8;     // (rows past the end: the last, never stored)
  const TA* ap[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) ap[m] = a + (size_t)min(m0 + m * 16 + r16, M - 1) * lda + kg * 8;
  f32x4_t acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // two batches of U steps in turn: while the MFMAs of one run, the loads of the other are on their way
  Eight<TW> wv[2][U];
  Eight<TA> av[2][U][MT];
  auto load = [&](int buf, int s) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      fetch8(wp + (s + u) * 32, wv[buf][u]);
#pragma unroll
      for (int m = 0; m < MT; ++m) fetch8(ap[m] + (s + u) * 32, av[buf][u][m]);
    }
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(value8(wv[buf][u], e), value8(av[buf][u][m], e), acc[m], 0, 0, 0);
  };
  const int batches = (end - begin) / U;
  if (batches > 0) load(0, begin);
  int b = 0;
  for (; b + 2 <= batches; b += 2) {
    load(1, begin + (b + 1) * U);
    multiply(0);
    if (b + 2 < batches) load(0, begin + (b + 2) * U);
    multiply(1);
  }
  if (b < batches) multiply(0);
  for (int s = begin + batches * U; s < end; ++s) {
    Eight<TW> wl;
    Eight<TA> al[MT];
    fetch8(wp + s * 32, wl);
#pragma unroll
    for (int m = 0; m < MT; ++m) fetch8(ap[m] + s * 32, al[m]);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(value8(wl, e), value8(al[m], e), acc[m], 0, 0, 0);
  }
  if (wave > 0) {
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wave - 1][m][lane] = acc[m];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int i = 0; i < WK - 1; ++i) acc[m] += red[i][m][lane];
    const int row = m0 + m * 16 + r16, n = n0 + kg * 4;
    if (row >= M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) c[(size_t)row * ldc + n + e] = from_f32<TC>(acc[m][e]);
  }
}

constexpr int kStreamRows = 64;       // rows of A that one streaming workgroup takes
constexpr int kCUs = 256;

static int ceil_div(int a, int b) { return (a + b - 1) / b; }

template <int WK, typename TA, typename TW, typename TC>
static void launch_stream(const TA* a, const TW* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc,
                          hipStream_t stream) {
  const dim3 block(64 * WK), grid(ceil_div(N, 16), ceil_div(M, kStreamRows));
#define ATOMA_STREAM(MT) \
  hipLaunchKernelGGL((f32_stream_kernel<MT, WK, TA, TW, TC>), grid, block, 0, stream, a, w, c, M, N, K, lda, ldw, ldc)
  if (M <= 16) ATOMA_STREAM(1);
  else if (M <= 32) ATOMA_STREAM(2);
  else ATOMA_STREAM(4);
#undef ATOMA_STREAM
}

template <typename TA, typename TW, typename TC>
static int launch(const TA* a, const TW* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  auto rows16 = [](const void* p, int ld, size_t size) { return ((uintptr_t)p | (ld * size)) % 16 == 0; };
  const bool aligned = rows16(a, lda, sizeof(TA)) && rows16(w, ldw, sizeof(TW));
  const int small = ceil_div(M, 64) * ceil_div(N, 64), large = ceil_div(M, 128) * ceil_div(N, 128);
  if (aligned && K % 32 == 0 && (M <= kStreamRows || small < kCUs)) {
    // eight waves a workgroup where N gives few of them, four else (the choice is N's alone: a row's sums do not depend
    // on how many rows there are beside it)
    if (N <= 4096) launch_stream<8>(a, w, c, M, N, K, lda, ldw, ldc, stream);
    else launch_stream<4>(a, w, c, M, N, K, lda, ldw, ldc, stream);
    ATOMA_LAUNCH_CHECK();
    return 0;
  }
  const bool vec = aligned && K % kF32Step == 0;
  const int T = large >= kCUs ? 128 : 64;
  if (ceil_div(M, T) > 65535) return ATOMA_ERR_SHAPE;
  const dim3 grid(ceil_div(N, T), ceil_div(M, T)), block(256);
#define ATOMA_TILE(T, V) \
  hipLaunchKernelGGL((f32_tile_kernel<T, V, TA, TW, TC>), grid, block, 0, stream, a, w, c, M, N, K, lda, ldw, ldc)
  if (T == 128 && vec) ATOMA_TILE(128, true);
  else if (T == 128) ATOMA_TILE(128, false);
  else if (vec) ATOMA_TILE(64, true);
  else ATOMA_TILE(64, false);
#undef ATOMA_TILE
  ATOMA_LAUNCH_CHECK();
  return 0;
}

template <typename TA, typename TW>
static int launch_c(const TA* a, const TW* w, void* c, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc,
                    hipStream_t stream) {
  if (c_dtype == kF32) return launch(a, w, (float*)c, M, N, K, lda, ldw, ldc, stream);
  if (c_dtype == kBF16) return launch(a, w, (bf16_t*)c, M, N, K, lda, ldw, ldc, stream);
  return ATOMA_ERR_DTYPE;
}

template <typename TA>
static int launch_w(const TA* a, const void* w, int w_dtype, void* c, int c_dtype, int M, int N, int K, int lda,
                    int ldw, int ldc, hipStream_t stream) {
  if (w_dtype == kF32) return launch_c<TA, float>(a, (const float*)w, c, c_dtype, M, N, K, lda, ldw, ldc, stream);
  if (w_dtype == kBF16) return launch_c<TA, bf16_t>(a, (const bf16_t*)w, c, c_dtype, M, N, K, lda, ldw, ldc, stream);
  return ATOMA_ERR_DTYPE;
}

extern "C" int atoma_gemm_generic(const void* a, int a_dtype, const void* w, int w_dtype, void* c, int c_dtype, int M,
                                  int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldc < N) return ATOMA_ERR_SHAPE;
  if ((M + 63) / 64 > 65535) return ATOMA_ERR_SHAPE;
  if (a_dtype == kF32) return launch_w<float>((const float*)a, w, w_dtype, c, c_dtype, M, N, K, lda, ldw, ldc, stream);
  if (a_dtype == kBF16)
    return launch_w<bf16_t>((const bf16_t*)a, w, w_dtype, c, c_dtype, M, N, K, lda, ldw, ldc, stream);
  return ATOMA_ERR_DTYPE;
}
