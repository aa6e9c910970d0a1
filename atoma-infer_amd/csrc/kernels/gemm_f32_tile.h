// One workgroup's tile of C = A * W^T in true float32 on the matrix cores: v_mfma_f32_16x16x4_f32, whose products and
// sums are float32 fused multiply-adds.  Shared by the general product and by the experts' one.
//
// A workgroup of four waves owns TM rows of A against TN rows of W (TM, TN: 64 or 128), each wave a quarter of both
// (2 x 2).  Both operands pass LDS, 32 values of K a step, widened to float32 on the way in, two buffers in turn: the
// next step's pieces wait in registers while this one is multiplied, one barrier a step.  A lane takes eight neighbouring
// values of K of a row with two 16-byte LDS loads and feeds them to eight MFMAs: lane group g (of 16 lanes) holds values
// 8 g .. 8 g + 7 of the step, and MFMA j sums the values 8 g + j, the same ones of A and of W.  Rows of LDS are
// 36 floats apart, so that the sixteen rows of a load fall on sixteen different quadruples of banks.
//
// The order of a sum.  The instruction adds its four products one after the other, g ascending, each a fused multiply-add
// (a test holds it to that).  So a step of 32 values of K is added in the order 8 g + j: j = 0 .. 7 outside, g = 0 .. 3
// inside.  The general product's K is cut into four or eight parts of whole steps, summed each from zero and then in order:
// that is how the kernel that streams the weight splits K over its waves, and every other kernel of the general product
// keeps to it, so that a row's sums are a function of K and N, whatever rows stand beside it and whichever kernel that makes.
#pragma once
#include "common.h"

namespace atoma {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kF32Step = 32, kF32Row = kF32Step + 4;

// The parts of K of a general product with N columns are 1 << f32_part_bits(N): eight where N gives a streaming kernel few
// workgroups, four else.  Then the first step of one of them.
__host__ __device__ __forceinline__ constexpr int f32_part_bits(int N) { return N <= 4096 ? 3 : 2; }
__host__ __device__ __forceinline__ constexpr int f32_part_begin(int steps, int part, int bits) { return (steps * part) >> bits; }

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

// total[i][j] (i: blocks of 16 rows of W, j: blocks of 16 rows of A, of this wave's quarter): lane l holds rows
// 4 (l / 16) .. + 3 of W's block against row l % 16 of A's.  row_a(r), row_w(r): the pointer to row r of the tile
// (of any row that can be read, for one past the end: its results are never stored); scale(r) multiplies row r of A.
// SPLIT: K is in 1 << bits parts (see above).
template <int TM, int TN, bool VEC, bool SPLIT, typename TA, typename TW, typename RowA, typename RowW, typename Scale>
__device__ __forceinline__ void f32_tile(float* __restrict__ lds, int K, int bits, RowA row_a, RowW row_w, Scale scale,
                                         f32x4_t (&total)[TN / 32][TM / 32]) {
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
  f32x4_t acc[TN / 32][TM / 32];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < TN / 32; ++i)
#pragma unroll
      for (int j = 0; j < TM / 32; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
#pragma unroll
  for (int i = 0; i < TN / 32; ++i)
#pragma unroll
    for (int j = 0; j < TM / 32; ++j) total[i][j] = acc[i][j];
  const int steps = (K + kF32Step - 1) / kF32Step;
  int part = 0, next = SPLIT ? f32_part_begin(steps, 1, bits) : steps;
  fetch(0);
  int buf = 0;
  for (int s = 0, k = 0; s < steps; ++s, k += kF32Step, buf ^= 1) {
    if constexpr (SPLIT) {
      if (s == next) {
#pragma unroll
        for (int i = 0; i < TN / 32; ++i)
#pragma unroll
          for (int j = 0; j < TM / 32; ++j) total[i][j] += acc[i][j];
        clear();
        // (parts without a step add nothing)
        do next = f32_part_begin(steps, ++part + 1, bits);
        while (next == s);
      }
    }
    float* const as = lds + buf * BUF;
    float* const ws = as + TM * kF32Row;
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      f32x4_t v = f32_wide(va[i]) * sa[i];
      if constexpr (!VEC) {      // (zeros beyond K, also times an infinite scale)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = k + k4 + e < K ? v[e] : 0.f;
      }
      *reinterpret_cast<f32x4_t*>(as + (r0 + i * 32) * kF32Row + k4) = v;
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) *reinterpret_cast<f32x4_t*>(ws + (r0 + i * 32) * kF32Row + k4) = f32_wide(vw[i]);
    __syncthreads();      // (the other buffer was last read before the barrier of the step before)
    if (k + kF32Step < K) fetch(k + kF32Step);
    const float* const aw = as + ((wave >> 1) * (TM / 2) + r16) * kF32Row + kg * 8;
    const float* const ww = ws + ((wave & 1) * (TN / 2) + r16) * kF32Row + kg * 8;
#pragma unroll
    for (int half = 0; half < 8; half += 4) {
      f32x4_t fa[TM / 32], fw[TN / 32];
#pragma unroll
      for (int j = 0; j < TM / 32; ++j) fa[j] = *reinterpret_cast<const f32x4_t*>(aw + j * 16 * kF32Row + half);
#pragma unroll
      for (int i = 0; i < TN / 32; ++i) fw[i] = *reinterpret_cast<const f32x4_t*>(ww + i * 16 * kF32Row + half);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TN / 32; ++i)
#pragma unroll
          for (int j = 0; j < TM / 32; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[i][e], fa[j][e], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < TN / 32; ++i)
#pragma unroll
    for (int j = 0; j < TM / 32; ++j) total[i][j] = SPLIT ? total[i][j] + acc[i][j] : acc[i][j];
}

// ---- float32 rows against a bfloat16 weight -----------------------------------------------------------------------------
// A float32 number is the sum of three bfloat16 numbers of its sign (24 bits of significand, eight at a time), so a product of
// float32 rows and a bfloat16 weight is three bfloat16 ones, whose products float32 holds exactly and whose sums the matrix cores
// keep in float32: 32 values of K take three instructions where they took eight of twice the length.  A step of 32 values is added as
// the weight times the first, the second and the third bfloat16 of each value, by v_mfma_f32_16x16x32_bf16 with lane group g holding
// values 8 g .. 8 g + 7; the parts of K are those above.  Every kernel of the general product keeps to that.
// Its error against 64-bit results is smaller than the float32 instruction's, which rounds after each of a step's values.  By that one / by
// this one, of the results' size, 200 rows, 4,096 columns, K of 2,048 and of 8,192: normal values 2.9e-7 / 1.9e-7 and 5.8e-7 / 3.5e-7,
// those of either sign and size e^(2 normal) 2.0e-7 / 1.4e-7 and 5.3e-7 / 2.8e-7, uniform from 0 to 1 9.0e-8 / 6.9e-8 and 1.6e-7 / 1.1e-7,
// 1 + 0.1 normal 8.8e-8 / 6.5e-8 and 1.6e-7 / 1.4e-7.
// But it has a direction, where the float32 instruction's average is below 2e-9: normal values' results are too low by 1.5e-8 (K of 2,048)
// to 5.7e-8 (8,192) of their size on average, whatever their own sign, and positive ones of parts of 1,024 values too high by up to 9e-8.
// What sums over such results adds that up.  And it grows where all products have one sign and a part's sum outgrows them by far: in parts
// of 1,280 values the two are even, in parts of 2,560 it is 1.9e-6 against 3.9e-7.  So parts longer than 1,024 values keep the float32
// instruction.
__host__ __device__ __forceinline__ constexpr bool split_product(int N, int K) { return K <= 1024 << f32_part_bits(N); }
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

struct Split8 { bf16x8_t p[3]; };

__device__ __forceinline__ uint32_t high_halves(float lo, float hi) {      // the upper sixteen bits of both
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302);
}
// Exact but for what lies below 2^-133 (bfloat16's smallest number).  An infinite value's second and third number are those of
// the largest finite one, so that its products stay infinities.  What is no number stays none: a payload in the lower half alone, which
// the first number loses, is that of a signalling one, and v_med3_f32, which is the least of its operands then, passes on such a one as
// the last of them (the test of these products holds it to that; with the value in front it would be the largest number's negative).
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  u32x4 h[3];
  float most = 3.402823466e38f;
  asm("" : "+s"(most));      // (constants would be moved behind the value)
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float r[2], t[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float v = __builtin_amdgcn_fmed3f(-most, most, x[i + e]);
      r[e] = v - __uint_as_float(__float_as_uint(v) & 0xffff0000u);
      t[e] = r[e] - __uint_as_float(__float_as_uint(r[e]) & 0xffff0000u);
    }
    h[0][i / 2] = high_halves(x[i], x[i + 1]);
    h[1][i / 2] = high_halves(r[0], r[1]);
    h[2][i / 2] = high_halves(t[0], t[1]);
  }
  Split8 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.p[q] = __builtin_bit_cast(bf16x8_t, h[q]);
  return s;
}

// The weight as the second and third numbers meet it: its infinities and NaN made the largest finite numbers (those numbers may
// be zero, and the first one's product has said what the sum is).
__device__ __forceinline__ bf16x8_t split_weight(bf16x8_t w) {
  typedef __attribute__((ext_vector_type(8))) short i16x8;
  typedef __attribute__((ext_vector_type(8))) unsigned short u16x8;
  const i16x8 a = __builtin_elementwise_min(__builtin_bit_cast(i16x8, w), (i16x8)(short)0x7f7f);
  return __builtin_bit_cast(bf16x8_t, __builtin_elementwise_min(__builtin_bit_cast(u16x8, a), (u16x8)(unsigned short)0xff7f));
}

// eight neighbouring values of K of one row, from k on; zeros from K on.  VEC: as in f32_load4, and the rows are aligned to 16 bytes
template <bool VEC>
__device__ __forceinline__ void split_load(const float* __restrict__ row, int k, int K, f32x4_t (&v)[2]) {
  if constexpr (VEC) {
    v[0] = *reinterpret_cast<const f32x4_t*>(row + k), v[1] = *reinterpret_cast<const f32x4_t*>(row + k + 4);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i >> 2][i & 3] = k + i < K ? row[k + i] : 0.f;
  }
}
template <bool VEC>
__device__ __forceinline__ void split_load(const bf16_t* __restrict__ row, int k, int K, uint4& v) {
  if constexpr (VEC) {
    v = *reinterpret_cast<const uint4*>(row + k);
  } else {
    uint16_t* const e = reinterpret_cast<uint16_t*>(&v);
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = k + i < K ? __builtin_bit_cast(uint16_t, row[k + i]) : (uint16_t)0;
  }
}
__device__ __forceinline__ Split8 split_of(const f32x4_t (&v)[2]) {
  const float x[8] = {v[0][0], v[0][1], v[0][2], v[0][3], v[1][0], v[1][1], v[1][2], v[1][3]};
  return split8(x);
}

// A row of a step in LDS: 64 bytes, 80 apart, so that the sixteen rows of a load fall on different banks.
constexpr int kSplitRow = 80;
// TM rows of A against TN rows of W by WM x WN waves; bytes of LDS: two buffers of A's three planes and W's rows
template <int TM_, int TN_, int WM_, int WN_, int ST_>
struct SplitTile {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, ST = ST_, THREADS = 64 * WM * WN;
  static constexpr int BM = TM / WM / 16, BN = TN / WN / 16;             // blocks of 16 of a wave
  static constexpr int PLANE = TM * kSplitRow, BUF = (3 * TM + TN) * kSplitRow, LDS = 2 * BUF;
  static_assert(TM * 4 % THREADS == 0 && TN * 4 % THREADS == 0 && LDS <= 160 * 1024, "");
};

// As f32_tile with SPLIT and no scale: total[i][j] of this wave's share (wave / WN of A's rows, wave % WN of W's).  A step's values
// are asked for ST + 1 steps ahead, wait in registers in ST sets in turn (two, and four where a wave's share leaves room), and are split
// and written to LDS beside the products of the step before theirs: one barrier a step.
template <typename C, bool VEC, typename RowA, typename RowW>
__device__ __forceinline__ void split_tile(char* __restrict__ lds, int K, int bits, RowA row_a, RowW row_w,
                                           f32x4_t (&total)[C::BN][C::BM]) {
  constexpr int PA = C::TM * 4 / C::THREADS, PW = C::TN * 4 / C::THREADS, RP = C::THREADS / 4;      // pieces of eight a thread moves
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int k8 = (tid & 3) * 8, r0 = tid >> 2;             // four threads a row of the step
  const float* pa[PA];
  const bf16_t* pw[PW];
#pragma unroll
  for (int i = 0; i < PA; ++i) pa[i] = row_a(r0 + i * RP);
#pragma unroll
  for (int i = 0; i < PW; ++i) pw[i] = row_w(r0 + i * RP);
  struct Stage { f32x4_t a[PA][2]; uint4 w[PW]; };
  const int steps = (K + kF32Step - 1) / kF32Step;
  auto fetch = [&](Stage& st, int s) {                     // (steps past the end: the last one again, which nobody multiplies)
    const int k = min(s, steps - 1) * kF32Step + k8;
#pragma unroll
    for (int i = 0; i < PA; ++i) split_load<VEC>(pa[i], k, K, st.a[i]);
#pragma unroll
    for (int i = 0; i < PW; ++i) split_load<VEC>(pw[i], k, K, st.w[i]);
  };
  auto put = [&](char* buf, const Stage& st) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
      const Split8 x = split_of(st.a[i]);
      bf16x8_t* const to = reinterpret_cast<bf16x8_t*>(buf + (r0 + i * RP) * kSplitRow + k8 * 2);
      to[0] = x.p[0], to[C::PLANE / 16] = x.p[1], to[2 * C::PLANE / 16] = x.p[2];
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) *reinterpret_cast<uint4*>(buf + 3 * C::PLANE + (r0 + i * RP) * kSplitRow + k8 * 2) = st.w[i];
  };
  f32x4_t acc[C::BN][C::BM];
#pragma unroll
  for (int i = 0; i < C::BN; ++i)
#pragma unroll
    for (int j = 0; j < C::BM; ++j) total[i][j] = acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int part = 0, next = f32_part_begin(steps, 1, bits);
  const int aw = (wave / C::WN * (C::TM / C::WM) + r16) * kSplitRow + kg * 16;
  const int ww = 3 * C::PLANE + (wave % C::WN * (C::TN / C::WN) + r16) * kSplitRow + kg * 16;
  // step s: its values lie in `now`; those of step s + 1 come in `st` and go to `then`
  auto step = [&](int s, const char* now, char* then, Stage& st) {
    if (s == next) {
#pragma unroll
      for (int i = 0; i < C::BN; ++i)
#pragma unroll
        for (int j = 0; j < C::BM; ++j) total[i][j] += acc[i][j], acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      // (parts without a step add nothing)
      do next = f32_part_begin(steps, ++part + 1, bits);
      while (next == s);
    }
    // (everybody has written this step's values and read those of the step before)
    lds_barrier();
    bf16x8_t fw[C::BN];
#pragma unroll
    for (int i = 0; i < C::BN; ++i) fw[i] = *reinterpret_cast<const bf16x8_t*>(now + ww + i * 16 * kSplitRow);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      bf16x8_t fa[C::BM];
#pragma unroll
      for (int j = 0; j < C::BM; ++j) fa[j] = *reinterpret_cast<const bf16x8_t*>(now + aw + q * C::PLANE + j * 16 * kSplitRow);
      if (q == 1) {
#pragma unroll
        for (int i = 0; i < C::BN; ++i) fw[i] = split_weight(fw[i]);
      }
#pragma unroll
      for (int i = 0; i < C::BN; ++i)
#pragma unroll
        for (int j = 0; j < C::BM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i], fa[j], acc[i][j], 0, 0, 0);
    }
    put(then, st);
    fetch(st, s + C::ST + 1);
  };
  Stage st[C::ST];
#pragma unroll
  for (int i = 0; i < C::ST; ++i) fetch(st[i], i);
  put(lds, st[0]);
  fetch(st[0], C::ST);
  for (int s = 0; s < steps; s += C::ST) {
#pragma unroll
    for (int i = 0; i < C::ST; ++i)
      if (s + i < steps) step(s + i, lds + (i & 1) * C::BUF, lds + (~i & 1) * C::BUF, st[(i + 1) % C::ST]);
  }
#pragma unroll
  for (int i = 0; i < C::BN; ++i)
#pragma unroll
    for (int j = 0; j < C::BM; ++j) total[i][j] += acc[i][j];
}

}  // namespace atoma
