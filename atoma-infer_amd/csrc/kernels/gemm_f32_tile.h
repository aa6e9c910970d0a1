// One workgroup's tile of C = A * W^T in true float32 on the matrix cores: v_mfma_f32_16x16x4_f32, whose products and
// sums are float32 fused multiply-adds.  Shared by the general product and by the experts' one.
//
// A workgroup of four waves owns TM rows of A against TN rows of W (TM, TN: 64 or 128), each wave a quarter of both
// (2 x 2).  Both operands pass LDS, 32 values of K a step, widened to float32 on the way in, two buffers in turn: the
// next step's pieces wait in registers while this one is multiplied, one barrier a step.  A lane takes four neighbouring
// values of K of a row with one 16-byte LDS load and feeds them to four MFMAs: lane group g (of 16 lanes) holds values
// 4 g .. 4 g + 3 of a run of 16, and MFMA j sums the runs' values 4 g + j, the same ones of A and of W.  Rows of LDS are
// 36 floats apart, so that the sixteen rows of a load fall on sixteen different quadruples of banks.
#pragma once
#include "common.h"

namespace atoma {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kF32Step = 32, kF32Row = kF32Step + 4;

// four neighbouring values of K of one row as they come from memory, from k on; zeros from K on.  VEC: rows are aligned to
// four values and K is a multiple of the step, so that no load stands under a condition (the compiler waits for such a
// load where its branches meet, and the next step's fetch would not run under this one's products).
template <typename T> struct F32Raw { f32x4_t v; };
template <> struct F32Raw<bf16_t> { uint2 v; };
template <bool VEC, typename T>
__device__ __forceinline__ F32Raw<T> f32_load4(const T* __restrict__ row, int k, int K) {
  F32Raw<T> r;
  if constexpr (VEC) {
    r.v = *reinterpret_cast<const decltype(r.v)*>(row + k);
  } else {
    T* const e = reinterpret_cast<T*>(&r.v);
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = k + i < K ? row[k + i] : from_f32<T>(0.f);
  }
  return r;
}
__device__ __forceinline__ f32x4_t f32_wide(const F32Raw<float>& r) { return r.v; }
__device__ __forceinline__ f32x4_t f32_wide(const F32Raw<bf16_t>& r) {
  return f32x4_t{__uint_as_float(r.v.x << 16), __uint_as_float(r.v.x & 0xffff0000u), __uint_as_float(r.v.y << 16),
                 __uint_as_float(r.v.y & 0xffff0000u)};
}

// acc[i][j] (i: blocks of 16 rows of W, j: blocks of 16 rows of A, of this wave's quarter): lane l holds rows
// 4 (l / 16) .. + 3 of W's block against row l % 16 of A's.  row_a(r), row_w(r): the pointer to row r of the tile
// (of any row that can be read, for one past the end: its results are never stored); scale(r) multiplies row r of A.
template <int TM, int TN, bool VEC, typename TA, typename TW, typename RowA, typename RowW, typename Scale>
__device__ __forceinline__ void f32_tile(float* __restrict__ lds, int K, RowA row_a, RowW row_w, Scale scale,
                                         f32x4_t (&acc)[TN / 32][TM / 32]) {
  constexpr int PA = TM * (kF32Step / 4) / 256, PW = TN * (kF32Step / 4) / 256;      // pieces of four a thread moves
  constexpr int BUF = (TM + TN) * kF32Row;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int k4 = (tid & 7) * 4, r0 = tid >> 3;             // eight threads a row of the step
  const TA* pa[PA];
  float sa[PA];
  const TW* pw[PW];
#pragma unroll
  for (int i = 0; i < PA; ++i) pa[i] = row_a(r0 + i * 32), sa[i] = scale(r0 + i * 32);
#pragma unroll
  for (int i = 0; i < PW; ++i) pw[i] = row_w(r0 + i * 32);
  F32Raw<TA> va[PA];
  F32Raw<TW> vw[PW];
  auto fetch = [&](int k) {
#pragma unroll
    for (int i = 0; i < PA; ++i) va[i] = f32_load4<VEC>(pa[i], k + k4, K);
#pragma unroll
    for (int i = 0; i < PW; ++i) vw[i] = f32_load4<VEC>(pw[i], k + k4, K);
  };
  fetch(0);
  int buf = 0;
  for (int k = 0; k < K; k += kF32Step, buf ^= 1) {
    float* const as = lds + buf * BUF;
    float* const ws = as + TM * kF32Row;
#pragma unroll
    for (int i = 0; i < PA; ++i) *reinterpret_cast<f32x4_t*>(as + (r0 + i * 32) * kF32Row + k4) = f32_wide(va[i]) * sa[i];
#pragma unroll
    for (int i = 0; i < PW; ++i) *reinterpret_cast<f32x4_t*>(ws + (r0 + i * 32) * kF32Row + k4) = f32_wide(vw[i]);
    __syncthreads();      // (the other buffer was last read before the barrier of the step before)
    if (k + kF32Step < K) fetch(k + kF32Step);
    const float* const aw = as + ((wave >> 1) * (TM / 2) + r16) * kF32Row + kg * 4;
    const float* const ww = ws + ((wave & 1) * (TN / 2) + r16) * kF32Row + kg * 4;
#pragma unroll
    for (int run = 0; run < kF32Step; run += 16) {
      f32x4_t fa[TM / 32], fw[TN / 32];
#pragma unroll
      for (int j = 0; j < TM / 32; ++j) fa[j] = *reinterpret_cast<const f32x4_t*>(aw + j * 16 * kF32Row + run);
#pragma unroll
      for (int i = 0; i < TN / 32; ++i) fw[i] = *reinterpret_cast<const f32x4_t*>(ww + i * 16 * kF32Row + run);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TN / 32; ++i)
#pragma unroll
          for (int j = 0; j < TM / 32; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[i][e], fa[j][e], acc[i][j], 0, 0, 0);
    }
  }
}

}  // namespace atoma
