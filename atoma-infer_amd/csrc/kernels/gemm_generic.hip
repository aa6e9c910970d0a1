// C[M, N] = A[M, K] * W[N, K]^T in true float32: products and sums are float32 fused multiply-adds (on the matrix
// cores' float32 instruction), or, for float32 rows against a bfloat16 weight, exact products of all of a value's bits
// with float32 sums; no reduced-precision mode.  A and W may be float32 or bfloat16 (widened exactly on
// load); C float32 or bfloat16.  Any M, N, K.  It is the product of the 32-bit path and the fallback for shapes the
// bfloat16 kernels refuse.
//
// Weights are [out, in] row-major as checkpoints store them (models/src/llama.rs:322-325), so both operands
// are contiguous along K.  Two kernels, each in two kinds:
//
//   f32_tile_kernel    tiles of 128 x 128 (64 x 64 where those would leave CUs idle) through LDS, see gemm_f32_tile.h.
//                      Bound by the matrix cores (a float32 MFMA has a sixteenth of the bfloat16 rate);
//   f32_stream_kernel  up to 64 rows of A a workgroup against 16 rows of W, which come straight from memory, once: K is
//                      split over the workgroup's waves, whose sums meet in LDS.  Bound by W's bytes up to 16 rows of A.
//                      It also takes more rows where tiles of 64 x 64 would be fewer than the CUs (four waves of a tile
//                      walk all of K, eight of a streaming workgroup an eighth of it each);
//   split_tile_kernel, split_stream_kernel, split_few_kernel (up to 24 rows)
//                      the same for float32 rows against a bfloat16 weight, which is the 32-bit path of a bfloat16 checkpoint:
//                      every float32 value as three bfloat16 ones (gemm_f32_tile.h), at three bfloat16 MFMAs for 32 values of K.
//                      Tiles are bound by what a step costs beside its MFMAs (splitting A, a trip through LDS, a barrier: 1.4 us for
//                      128 x 256, of which the MFMAs are 0.7), streaming workgroups by W's bytes and the splitting.
//
// Measured on MI355X, float32 rows against bfloat16 weights, us by the float32 MFMA / by three bfloat16 ones: gate-up of Llama 1B
// (16,384 x 2,048) with 836 rows 568 / 175, with 64 rows 73 / 32, with 4 rows 17.3 / 13.4; its down product (2,048 x 8,192) with 836
// rows 317 / 155, with 4 rows 16.4 / 11.4; q, k, v (3,072 x 2,048) with 836 rows 123 / 60; the head (128,256 x 2,048) with 4 rows 114 / 87, with 64
// rows 557 / 153.
//
// All sum an output's K products in the order that gemm_f32_tile.h states, a function of (N, K) alone: a row's
// result depends neither on its place nor on the rows beside it.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "cache_layout.h"
#include "gate_act.h"
#include "gemm_f32_tile.h"

using namespace atoma;

// Results n .. n + 3 of a row of C; aligned: a row's quadruples are (16 or 8 bytes in one store where all four are there: with
// K of 36 the stores are most of the time: 2,048 x 4,096 results 33 -> 23.5 us, 25.4 by the kernel of vector multiply-adds)
__device__ __forceinline__ void put4(float* row, int n, int N, bool aligned, f32x4_t v) {
  if (aligned && n + 4 <= N) {
    *reinterpret_cast<f32x4_t*>(row + n) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) row[n + e] = v[e];
}
__device__ __forceinline__ void put4(bf16_t* row, int n, int N, bool aligned, f32x4_t v) {
  if (aligned && n + 4 <= N) {
    *reinterpret_cast<uint2*>(row + n) =
        make_uint2(f32_to_bf16_bits(v[0]) | (uint32_t)f32_to_bf16_bits(v[1]) << 16,
                   f32_to_bf16_bits(v[2]) | (uint32_t)f32_to_bf16_bits(v[3]) << 16);
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < N) row[n + e] = from_f32<bf16_t>(v[e]);
}
template <typename TC> __device__ __forceinline__ bool aligned4(const TC* c, int ldc) {
  return ldc % 4 == 0 && (uintptr_t)c % (4 * sizeof(TC)) == 0;
}

template <int T, bool VEC, typename TA, typename TW, typename TC>
__global__ void __launch_bounds__(256)
f32_tile_kernel(const TA* __restrict__ a, const TW* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                int ldw, int ldc) {
  __shared__ __attribute__((aligned(16))) float lds[2 * 2 * T * kF32Row];
  const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
  f32x4_t acc[T / 32][T / 32];
  f32_tile<T, T, VEC, true, TA, TW>(
      lds, K, f32_part_bits(N), [&](int r) { return a + (size_t)min(m0 + r, M - 1) * lda; },
      [&](int r) { return w + (size_t)min(n0 + r, N - 1) * ldw; }, [](int) { return 1.f; }, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool aligned = aligned4(c, ldc);
#pragma unroll
  for (int j = 0; j < T / 32; ++j) {
    const int m = m0 + (wave >> 1) * (T / 2) + j * 16 + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < T / 32; ++i) {
      const int n = n0 + (wave & 1) * (T / 2) + i * 16 + (lane >> 4) * 4;
      put4(c + (size_t)m * ldc, n, N, aligned, acc[i][j]);
    }
  }
}

// the same for float32 rows against a bfloat16 weight
template <typename C, bool VEC, typename TC>
__global__ void __launch_bounds__(C::THREADS, 2)
split_tile_kernel(const float* __restrict__ a, const bf16_t* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                  int ldw, int ldc) {
  extern __shared__ __attribute__((aligned(16))) char split_lds[];
  const int m0 = blockIdx.y * C::TM, n0 = blockIdx.x * C::TN;
  f32x4_t acc[C::BN][C::BM];
  split_tile<C, VEC>(
      split_lds, K, f32_part_bits(N), [&](int r) { return a + (size_t)min(m0 + r, M - 1) * lda; },
      [&](int r) { return w + (size_t)min(n0 + r, N - 1) * ldw; }, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool aligned = aligned4(c, ldc);
#pragma unroll
  for (int j = 0; j < C::BM; ++j) {
    const int m = m0 + wave / C::WN * (C::TM / C::WM) + j * 16 + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < C::BN; ++i) {
      const int n = n0 + wave % C::WN * (C::TN / C::WN) + i * 16 + (lane >> 4) * 4;
      put4(c + (size_t)m * ldc, n, N, aligned, acc[i][j]);
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
  constexpr int BITS = WK == 8 ? 3 : 2;
  static_assert(WK == 1 << BITS, "a wave a part of K");
  constexpr int U = MT == 1 ? 4 : 2;       // steps whose loads are in flight together
  __shared__ f32x4_t red[WK - 1][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
  const int steps = K / 32, begin = f32_part_begin(steps, wave, BITS), end = f32_part_begin(steps, wave + 1, BITS);
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
    put4(c + (size_t)row * ldc, n, N, aligned4(c, ldc), acc[m]);
  }
}

// The same for float32 rows against a bfloat16 weight: a step is 32 values of K, three instructions for each block of 16 rows of A
// and of W.  RT blocks of W a wave share the split of A's values, which takes as long as four blocks' instructions.
template <int MT, int RT, int WK, typename TC>
__global__ void __launch_bounds__(64 * WK)
split_stream_kernel(const float* __restrict__ a, const bf16_t* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                    int ldw, int ldc) {
  constexpr int BITS = WK == 8 ? 3 : 2;
  static_assert(WK == 1 << BITS, "a wave a part of K");
  constexpr int U = MT == 1 && RT == 1 ? 4 : 2;       // steps whose loads are in flight together
  __shared__ f32x4_t red[WK - 1][RT][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * (16 * RT), m0 = blockIdx.y * (16 * MT);
  const int steps = K / 32, begin = f32_part_begin(steps, wave, BITS), end = f32_part_begin(steps, wave + 1, BITS);
  const bf16_t* wp[RT];                                    // (rows past the end: the last, never stored)
#pragma unroll
  for (int i = 0; i < RT; ++i) wp[i] = w + (size_t)min(n0 + i * 16 + r16, N - 1) * ldw + kg * 8;
  const float* ap[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) ap[m] = a + (size_t)min(m0 + m * 16 + r16, M - 1) * lda + kg * 8;
  f32x4_t acc[RT][MT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[i][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  struct Step { bf16x8_t w[RT]; f32x4_t a[MT][2]; };
  auto load = [&](Step& x, int s) {
#pragma unroll
    for (int i = 0; i < RT; ++i) x.w[i] = *reinterpret_cast<const bf16x8_t*>(wp[i] + s * 32);
#pragma unroll
    for (int m = 0; m < MT; ++m) split_load<true>(ap[m], s * 32, K, x.a[m]);
  };
  auto multiply = [&](Step& x) {
    Split8 p[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) p[m] = split_of(x.a[m]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      if (q == 1) {
#pragma unroll
        for (int i = 0; i < RT; ++i) x.w[i] = split_weight(x.w[i]);
      }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[i][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.w[i], p[m].p[q], acc[i][m], 0, 0, 0);
    }
  };
  // two batches of U steps in turn: while the MFMAs of one run, the loads of the other are on their way
  Step x[2][U];
  const int batches = (end - begin) / U;
  auto fetch = [&](int buf, int b) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(x[buf][u], begin + b * U + u);
  };
  auto take = [&](int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(x[buf][u]);
  };
  if (batches > 0) fetch(0, 0);
  int b = 0;
  for (; b + 2 <= batches; b += 2) {
    fetch(1, b + 1);
    take(0);
    if (b + 2 < batches) fetch(0, b + 2);
    take(1);
  }
  if (b < batches) take(0);
  for (int s = begin + batches * U; s < end; ++s) {
    load(x[0][0], s);
    multiply(x[0][0]);
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m) red[wave - 1][i][m][lane] = acc[i][m];
  }
  __syncthreads();
  if (wave > 0) return;
  const bool aligned = aligned4(c, ldc);
#pragma unroll
  for (int i = 0; i < RT; ++i) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int q = 0; q < WK - 1; ++q) acc[i][m] += red[q][i][m][lane];
      const int row = m0 + m * 16 + r16, n = n0 + i * 16 + kg * 4;
      if (row >= M) continue;
      put4(c + (size_t)row * ldc, n, N, aligned, acc[i][m]);
    }
  }
}

// The same for up to 4 RW rows of A, 4 to 16, behind FULL blocks of 16 (none or one): sixteen lanes split a row's values of four steps and
// hand them to the others through LDS, so that no lane splits what another splits too (every wave has its own corner of LDS, which it
// fills and reads in order, with more than eight rows half a batch at a time).  A full block's rows are each lane's own.
// END: what leaves.  kPlain: the sums; kGated: act(gate) * up [M][ldc] of a weight in blocks of 16 gate rows and their 16 up rows, a wave
// having one of each (RT 2); kRotated: q rotated [M][ldc] and k, v in the float32 cache, the rows of q and k heads in pair order (columns 2 i and
// 2 i + 1 are the members of pair i).  The sums are those of the other kernels, and the ends compute as the activation's and the rotation's own
// kernels do, so the bits are theirs; what is saved is a launch.  Llama 1B sizes in float32, four layers, four requests: a pass of prompts and 16 decoded tokens 8.03 -> 7.76 ms.
enum FewEnd : int { kPlain, kGated, kRotated };
struct FewArgs {
  GateAct act;
  const int32_t* positions;      // [M]
  const float* cos_t;            // [positions, hd / 2]
  const float* sin_t;
  float* kcache;                 // [pages, nkv, page_size * hd] tiles
  float* vcache;
  const int32_t* slot_mapping;   // [M]; negative: no cache write for the row
  int page_size, nh, nkv, hd;
};
// outputs n .. n + 3 of a row of the fused q, k, v projection (n a multiple of 4, hd too: one head)
__device__ __forceinline__ void rotate_store4(const FewArgs& f, float* __restrict__ q_row, int n, int pos, int slot, f32x4_t v) {
  const int head = n / f.hd, d = n - head * f.hd, half = f.hd >> 1;
  const int page = slot >= 0 ? slot / f.page_size : 0, off = slot >= 0 ? slot % f.page_size : 0;
  if (head >= f.nh + f.nkv) {
    if (slot < 0) return;
    float* const tile = f.vcache + ((size_t)page * f.nkv + (head - f.nh - f.nkv)) * f.hd * f.page_size;
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[value_offset(d + e, off, f.hd, f.page_size)] = v[e];
    return;
  }
  const bool is_k = head >= f.nh;
  if (is_k && slot < 0) return;
  float* const ktile = is_k ? f.kcache + ((size_t)page * f.nkv + (head - f.nh)) * f.page_size * f.hd : nullptr;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int i = (d >> 1) + p;
    const float c = f.cos_t[(size_t)pos * half + i], sv = f.sin_t[(size_t)pos * half + i];
    const float x1 = v[2 * p], x2 = v[2 * p + 1];
    const float o1 = fmaf(x1, c, -(x2 * sv)), o2 = fmaf(x1, sv, x2 * c);      // (as the compiler writes the rotation's own kernel)
    if (is_k) {
      ktile[key_offset(off, i, f.page_size)] = o1;
      ktile[key_offset(off, i + half, f.page_size)] = o2;
    } else {
      q_row[head * f.hd + i] = o1;
      q_row[head * f.hd + i + half] = o2;
    }
  }
}

template <int FULL, int RW, int RT, int WK, typename TC, int END = kPlain>
__global__ void __launch_bounds__(64 * WK)
split_few_kernel(const float* __restrict__ a, const bf16_t* __restrict__ w, TC* __restrict__ c, int M, int N, int K, int lda,
                 int ldw, int ldc, FewArgs few) {
  constexpr int BITS = WK == 8 ? 3 : 2, U = 4, H = RW > 2 ? U / 2 : U;      // steps of a batch, and at a time in LDS
  static_assert(WK == 1 << BITS, "a wave a part of K");
  __shared__ f32x4_t red[WK - 1][FULL + 1][RT][64];
  __shared__ bf16x8_t thirds[WK][3][RW * 4][H * 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * (16 * RT);
  const int steps = K / 32, begin = f32_part_begin(steps, wave, BITS), end = f32_part_begin(steps, wave + 1, BITS);
  const bf16_t* wp[RT];                                    // (rows past the end: the last, never stored)
#pragma unroll
  for (int i = 0; i < RT; ++i) wp[i] = w + (size_t)min(n0 + i * 16 + r16, N - 1) * ldw + kg * 8;
  const float* ap[RW];                                     // lane l splits values 8 (l % 16) .. + 7 of a batch, of rows l / 16 + 4 r
#pragma unroll
  for (int r = 0; r < RW; ++r) ap[r] = a + (size_t)min(FULL * 16 + kg + r * 4, M - 1) * lda + r16 * 8;
  const float* own[FULL + 1];                              // its own values of a step
#pragma unroll
  for (int m = 0; m <= FULL; ++m) own[m] = a + (size_t)min(m * 16 + r16, M - 1) * lda + kg * 8;
  int pos = 0, slot = -1;                                  // (asked for now: a trip to memory less behind the sums)
  if constexpr (END == kRotated) {
    static_assert(FULL == 0, "a lane a row");
    pos = few.positions[min(r16, M - 1)];
    slot = few.slot_mapping[min(r16, M - 1)];
  }
  f32x4_t acc[FULL + 1][RT];
#pragma unroll
  for (int m = 0; m <= FULL; ++m)
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[m][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  struct Batch { bf16x8_t w[U][RT]; f32x4_t full[U][FULL + 1][2], a[RW][2]; };
  auto fetch = [&](Batch& x, int s) {
#pragma unroll
    for (int r = 0; r < RW; ++r) split_load<true>(ap[r], s * 32, K, x.a[r]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < RT; ++i) x.w[u][i] = *reinterpret_cast<const bf16x8_t*>(wp[i] + (s + u) * 32);
#pragma unroll
      for (int m = 0; m < FULL; ++m) split_load<true>(own[m], (s + u) * 32, K, x.full[u][m]);
    }
  };
  const int row = r16 % (RW * 4);
  auto add = [&](bf16x8_t (&wv)[RT], const Split8 (&p)[FULL + 1]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      if (q == 1) {
#pragma unroll
        for (int i = 0; i < RT; ++i) wv[i] = split_weight(wv[i]);
      }
#pragma unroll
      for (int m = 0; m <= FULL; ++m)
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i], p[m].p[q], acc[m][i], 0, 0, 0);
    }
  };
  auto take = [&](Batch& x) {
    Split8 t[H < U ? RW : 1];
    auto put = [&](const Split8& v, int r) {
#pragma unroll
      for (int q = 0; q < 3; ++q) thirds[wave][q][kg + r * 4][r16 % (H * 4)] = v.p[q];
    };
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      if constexpr (H < U) t[r] = split_of(x.a[r]);
      else put(split_of(x.a[r]), r);
    }
#pragma unroll
    for (int h = 0; h < U; h += H) {
      if (H < U && r16 / (H * 4) == h / H) {
#pragma unroll
        for (int r = 0; r < RW; ++r) put(t[r], r);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int u = h; u < h + H; ++u) {
        Split8 p[FULL + 1];
#pragma unroll
        for (int m = 0; m < FULL; ++m) p[m] = split_of(x.full[u][m]);
#pragma unroll
        for (int q = 0; q < 3; ++q) p[FULL].p[q] = thirds[wave][q][row][(u - h) * 4 + kg];
        add(x.w[u], p);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  // two batches in turn: while the MFMAs of one run, the loads of the other are on their way
  Batch x[2];
  const int batches = (end - begin) / U;
  if (batches > 0) fetch(x[0], begin);
  int b = 0;
  for (; b + 2 <= batches; b += 2) {
    fetch(x[1], begin + (b + 1) * U);
    take(x[0]);
    if (b + 2 < batches) fetch(x[0], begin + (b + 2) * U);
    take(x[1]);
  }
  if (b < batches) take(x[0]);
  for (int s = begin + batches * U; s < end; ++s) {        // (steps that fill no batch: every lane its own)
    f32x4_t v[FULL + 1][2];
    bf16x8_t wv[RT];
#pragma unroll
    for (int m = 0; m <= FULL; ++m) split_load<true>(own[m], s * 32, K, v[m]);
#pragma unroll
    for (int i = 0; i < RT; ++i) wv[i] = *reinterpret_cast<const bf16x8_t*>(wp[i] + s * 32);
    Split8 p[FULL + 1];
#pragma unroll
    for (int m = 0; m <= FULL; ++m) p[m] = split_of(v[m]);
    add(wv, p);
  }
  if (wave > 0) {
#pragma unroll
    for (int m = 0; m <= FULL; ++m)
#pragma unroll
      for (int i = 0; i < RT; ++i) red[wave - 1][m][i][lane] = acc[m][i];
  }
  __syncthreads();
  if (wave > 0) return;
  const bool aligned = aligned4(c, ldc);
#pragma unroll
  for (int m = 0; m <= FULL; ++m) {
    if (m * 16 + r16 >= M) continue;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
      for (int q = 0; q < WK - 1; ++q) acc[m][i] += red[q][m][i][lane];
      if constexpr (END == kPlain) put4(c + (size_t)(m * 16 + r16) * ldc, n0 + i * 16 + kg * 4, N, aligned, acc[m][i]);
      else if constexpr (END == kRotated)
        if (n0 + i * 16 < N) rotate_store4(few, c + (size_t)r16 * ldc, n0 + i * 16 + kg * 4, pos, slot, acc[m][i]);
    }
    if constexpr (END == kGated) {
      static_assert(RT == 2 && FULL == 0, "gate and up in a wave");
      f32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = gated(acc[m][0][e], acc[m][1][e], few.act);
      put4(c + (size_t)r16 * ldc, n0 / 2 + kg * 4, N / 2, aligned, o);
    }
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

template <int FULL, int RW, int RT, typename TC>
static int launch_split_few(const float* a, const bf16_t* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  const dim3 grid(ceil_div(N, 16 * RT));
  // (a wave a part of K)
  if constexpr (RT == 1) {
    if (FULL > 0 || RW > 2 || f32_part_bits(N) == 3) {      // (of many columns only up to eight rows come here)
      hipLaunchKernelGGL((split_few_kernel<FULL, RW, RT, 8, TC>), grid, dim3(512), 0, stream, a, w, c, M, N, K, lda, ldw, ldc, FewArgs{});
      ATOMA_LAUNCH_CHECK();
      return 0;
    }
  }
  if constexpr (FULL == 0 && RW <= 2) {
    hipLaunchKernelGGL((split_few_kernel<FULL, RW, RT, 4, TC>), grid, dim3(256), 0, stream, a, w, c, M, N, K, lda, ldw, ldc, FewArgs{});
    ATOMA_LAUNCH_CHECK();
  }
  return 0;
}

template <int MT, int RT, typename TC>
static int launch_split_stream(const float* a, const bf16_t* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc,
                               hipStream_t stream) {
  const dim3 grid(ceil_div(N, 16 * RT), ceil_div(M, 16 * MT));
  // (a wave a part of K)
  if constexpr (RT <= 2) {
    if (f32_part_bits(N) == 3) {
      hipLaunchKernelGGL((split_stream_kernel<MT, RT, 8, TC>), grid, dim3(512), 0, stream, a, w, c, M, N, K, lda, ldw, ldc);
      ATOMA_LAUNCH_CHECK();
      return 0;
    }
  }
  hipLaunchKernelGGL((split_stream_kernel<MT, RT, 4, TC>), grid, dim3(256), 0, stream, a, w, c, M, N, K, lda, ldw, ldc);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

template <typename C, bool VEC, typename TC>
static int launch_split_tile(const float* a, const bf16_t* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  if (ceil_div(M, C::TM) > 65535) return ATOMA_ERR_SHAPE;
  // (every device that the kernel is launched on has its own setting)
  const hipError_t e = hipFuncSetAttribute((const void*)split_tile_kernel<C, VEC, TC>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  if (e != hipSuccess) return (int)e;
  hipLaunchKernelGGL((split_tile_kernel<C, VEC, TC>), dim3(ceil_div(N, C::TN), ceil_div(M, C::TM)), dim3(C::THREADS), C::LDS, stream,
                     a, w, c, M, N, K, lda, ldw, ldc);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// microseconds that tiles of C take: a step with one of them a CU, a round over the CUs, and as many as there are (fitted to 420
// products of 17 to 2,048 rows, 512 to 128,256 columns and K of 1,024 to 8,192, each tile within a quarter)
template <typename C>
static float split_tile_us(int M, int N, int K, float fixed, float one, float round, float each) {
  const float tiles = (float)ceil_div(M, C::TM) * ceil_div(N, C::TN) / kCUs;
  return fixed + ceil_div(K, kF32Step) * std::max({one, round * std::ceil(tiles), each * tiles});
}

// Which kernel takes float32 rows against a bfloat16 weight; whichever does, the results are the same bits.  Streaming workgroups of
// few blocks are the quickest as long as each has a CU (64 rows, 2,048 x 2,048: 10.3 us by one block of rows and two of the weight,
// 14.4 by two and two, 20.4 by four and one, 29.4 by tiles), so the first of the combinations below that is one round over
// the CUs; with more than 4,096 columns a workgroup has four waves and takes up to four blocks of each.  Beyond, tiles.
template <typename TC>
static int launch_split(const float* a, const bf16_t* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc, bool aligned,
                        hipStream_t stream) {
  const bool vec = aligned && K % kF32Step == 0, wide = f32_part_bits(N) == 2;
#define ATOMA_STREAM(MT, RT) return launch_split_stream<MT, RT>(a, w, c, M, N, K, lda, ldw, ldc, stream)
  if (vec) {
    auto round = [&](int mt, int rt, int most) { return (int64_t)ceil_div(N, 16 * rt) * ceil_div(M, 16 * mt) <= most; };
    // (up to eight rows the splitting is shared: 4 rows, 2,048 x 8,192 16.5 -> 11.4 us, 28,672 x 4,096 53 -> 41, the head of Llama 1B 101 -> 87;
    // two blocks of the weight against one, 4 rows: 5,120 x 3,072 9.3 and 10.0, 28,672 x 4,096 43.6 and 41.1)
#define ATOMA_FEW(FULL, RW, RT) return launch_split_few<FULL, RW, RT>(a, w, c, M, N, K, lda, ldw, ldc, stream)
    if (M <= 4) {
      if (!wide || (N > 16384 && N < 65536)) ATOMA_FEW(0, 1, 1);
      ATOMA_FEW(0, 1, 2);
    }
    if (M <= 8 && wide) ATOMA_FEW(0, 2, 2);
    if (M <= 8 && (M > 6 || K > 4096)) ATOMA_FEW(0, 2, 1);      // (5 rows, 2,048 x 2,048: 6.0 against 5.5 by the kernel below)
    if (!wide) {
      // (up to sixteen rows of long K likewise: 9 rows, 4,096 x 8,192 21.1 -> 18.8 us, x 4,096 11.5 -> 11.1, but x 3,584 10.3 -> 11.2; 16 rows,
      // x 8,192 24.9 -> 22.6, 13 of x 5,120 16.2 -> 16.1, but of x 4,096 12.8 -> 13.1)
      if (M <= 12 && K >= 4096) ATOMA_FEW(0, 3, 1);
      if (M <= 16 && K >= 5120) ATOMA_FEW(0, 4, 1);
      if (round(1, 1, kCUs)) ATOMA_STREAM(1, 1);
      // (a block of sixteen rows and up to eight behind it, against two blocks: 17 rows, 4,096 x 8,192 25.9 and 29.3 us, x 3,072 11.9 and 13.7, x
      // 1,024 5.35 and 5.65, x 768 4.94 and 4.67; 24 rows, against one block and two of the weight: 29.3 and 31.3, 13.5 and 13.7, 5.74 and 5.84)
      if (M <= 20 && K >= 1024) ATOMA_FEW(1, 1, 1);
      if (M <= 24 && K >= 1024) ATOMA_FEW(1, 2, 1);
      if (M <= 20) ATOMA_STREAM(2, 1);
      if (round(1, 2, kCUs)) ATOMA_STREAM(1, 2);
      if (round(2, 2, 320)) ATOMA_STREAM(2, 2);
      if (round(4, 2, kCUs)) ATOMA_STREAM(4, 2);
#undef ATOMA_FEW
    } else if (M <= 16) {
      if (N <= 8192) ATOMA_STREAM(1, 2);      // (16 rows, 8,192 x 4,096: 18.8 us, 26.9 by four blocks; 28,672 x 4,096: 65.7 and 57.8)
      ATOMA_STREAM(1, 4);
    } else {
      if (round(2, 2, kCUs)) ATOMA_STREAM(2, 2);
      if (round(1, 4, kCUs)) ATOMA_STREAM(1, 4);
      if (round(2, 4, kCUs) || (M <= 32 && N <= 65536)) ATOMA_STREAM(2, 4);
      if (round(4, 4, kCUs)) ATOMA_STREAM(4, 4);
    }
  }
#undef ATOMA_STREAM
  using Large = SplitTile<128, 256, 2, 4, 2>;
  using Middle = SplitTile<64, 128, 2, 2, 4>;
  using Small = SplitTile<64, 64, 2, 2, 2>;
#define ATOMA_TILE(C)                                                                                  \
  return vec ? launch_split_tile<C, true>(a, w, c, M, N, K, lda, ldw, ldc, stream)                    \
             : launch_split_tile<C, false>(a, w, c, M, N, K, lda, ldw, ldc, stream)
  const float large = split_tile_us<Large>(M, N, K, 7.17f, 1.03f, 0.3f, 1.58f), middle = split_tile_us<Middle>(M, N, K, 3.79f, 0.57f, 0.44f, 0.51f),
              small = split_tile_us<Small>(M, N, K, 2.7f, 0.43f, 0.31f, 0.2f);
  if (large <= std::min(middle, small)) ATOMA_TILE(Large);
  if (middle <= small) ATOMA_TILE(Middle);
  ATOMA_TILE(Small);
#undef ATOMA_TILE
}

template <typename TA, typename TW, typename TC>
static int launch(const TA* a, const TW* w, TC* c, int M, int N, int K, int lda, int ldw, int ldc, hipStream_t stream) {
  auto rows16 = [](const void* p, int ld, size_t size) { return ((uintptr_t)p | (ld * size)) % 16 == 0; };
  const bool aligned = rows16(a, lda, sizeof(TA)) && rows16(w, ldw, sizeof(TW));
  if constexpr (std::is_same_v<TA, float> && std::is_same_v<TW, bf16_t>) {
    if (split_product(N, K)) return launch_split(a, w, c, M, N, K, lda, ldw, ldc, aligned, stream);
  }
  const int small = ceil_div(M, 64) * ceil_div(N, 64), large = ceil_div(M, 128) * ceil_div(N, 128);
  if (aligned && K % 32 == 0 && (M <= kStreamRows || small < kCUs)) {
    // (a wave a part of K)
    if (f32_part_bits(N) == 3) launch_stream<8>(a, w, c, M, N, K, lda, ldw, ldc, stream);
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

// Whether products of up to eight float32 rows against a bfloat16 weight [N, K] have the two ends below.  gated: only weights of more than
// 4,096 rows, whose workgroups have a block of gate rows and one of up rows each; a narrower one's have a block of sixteen, so that there
// are enough of them.
extern "C" int atoma_gemm_few_takes(int M, int N, int K, int gated) {
  return M > 0 && M <= 8 && N > 0 && K > 0 && K % kF32Step == 0 && split_product(N, K) && N % (gated ? 32 : 16) == 0 &&
         (!gated || f32_part_bits(N) == 2);
}

template <int END>
static int launch_few_end(const float* a, const bf16_t* w, float* c, int M, int N, int K, int lda, int ldw, int ldc, const FewArgs& few, hipStream_t stream) {
#define ATOMA_FEW(RW, RT, WK)                                                                                                          \
  hipLaunchKernelGGL((split_few_kernel<0, RW, RT, WK, float, END>), dim3(ceil_div(N, 16 * RT)), dim3(64 * WK), 0, stream, a, w, c, M, N, K, \
                     lda, ldw, ldc, few)
  if (f32_part_bits(N) == 2) {
    if (M <= 4) ATOMA_FEW(1, 2, 4);
    else ATOMA_FEW(2, 2, 4);
  } else if constexpr (END == kRotated) {
    if (M <= 4) ATOMA_FEW(1, 1, 8);
    else ATOMA_FEW(2, 1, 8);
  } else {
    return ATOMA_ERR_SHAPE;
  }
#undef ATOMA_FEW
  ATOMA_LAUNCH_CHECK();
  return 0;
}

static bool few_fits(const void* a, const void* w, const void* c, int K, int lda, int ldw) {
  return lda >= K && ldw >= K && lda % 4 == 0 && ldw % 8 == 0 && (((uintptr_t)a | (uintptr_t)w | (uintptr_t)c) & 15) == 0;
}

// c [M, N / 2] = act(gate) * up of a [M <= 8, K] float32 times w [N, K] bfloat16 transposed, w in blocks of 16 gate rows and their 16 up rows.
extern "C" int atoma_gemm_few_gated(const float* a, const void* w, float* c, int M, int N, int K, int lda, int ldw, int ldc, int kind, float limit,
                                    float slope, hipStream_t stream) {
  if (M <= 0) return 0;
  if (!atoma_gemm_few_takes(M, N, K, 1) || !few_fits(a, w, c, K, lda, ldw) || ldc < N / 2 || !gate_act_ok(kind, limit)) return ATOMA_ERR_SHAPE;
  FewArgs few{};
  few.act = GateAct{kind, limit, slope};
  return launch_few_end<kGated>(a, (const bf16_t*)w, c, M, N, K, lda, ldw, ldc, few, stream);
}

// q_out [M, nh hd] rotated, k (rotated) and v in the float32 cache, of a [M <= 8, K] float32 times the fused q, k, v weight in pair order.
extern "C" int atoma_gemm_few_rotated(const float* a, const void* w, float* q_out, int M, int N, int K, int lda, int ldw, int ldq,
                                      const int32_t* positions, const float* cos_t, const float* sin_t, float* kcache, float* vcache,
                                      const int32_t* slot_mapping, int page_size, int nh, int nkv, int hd, hipStream_t stream) {
  if (M <= 0) return 0;
  if (!atoma_gemm_few_takes(M, N, K, 0) || !few_fits(a, w, q_out, K, lda, ldw) || nh <= 0 || nkv <= 0 || hd <= 0 || hd % 16 || N != (nh + 2 * nkv) * hd ||
      ldq < nh * hd || page_size <= 0 || !positions || !cos_t || !sin_t || !kcache || !vcache || !slot_mapping)
    return ATOMA_ERR_SHAPE;
  const FewArgs few{GateAct{0, 0.f, 0.f}, positions, cos_t, sin_t, kcache, vcache, slot_mapping, page_size, nh, nkv, hd};
  return launch_few_end<kRotated>(a, (const bf16_t*)w, q_out, M, N, K, lda, ldw, ldq, few, stream);
}
