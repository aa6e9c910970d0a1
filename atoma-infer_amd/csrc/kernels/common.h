// Shared device helpers for the gfx950 kernels: bfloat16 bit conversions, wave and block reductions,
// element-type dispatch.  Wavefronts are 64 lanes wide throughout.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace atoma {

constexpr int kWave = 64;

// bfloat16 is carried as its 16 raw bits.
struct bf16_t {
  uint16_t bits;
};

__device__ __host__ __forceinline__ float bf16_bits_to_f32(uint16_t b) {
  union { uint32_t u; float f; } v;
  v.u = ((uint32_t)b) << 16;
  return v.f;
}

// round to nearest, ties to even; NaN stays NaN
__device__ __host__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  union { uint32_t u; float f; } v;
  v.f = f;
  if ((v.u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((v.u >> 16) | 0x0040u);
  uint32_t lsb = (v.u >> 16) & 1u;
  v.u += 0x7fffu + lsb;
  return (uint16_t)(v.u >> 16);
}

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return bf16_bits_to_f32(v.bits); }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) {
  bf16_t r;
  r.bits = f32_to_bf16_bits(v);
  return r;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// A barrier for what passes LDS: unlike __syncthreads it does not wait for the wave's loads from and stores to memory.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Sum over a block of NWAVES*64 threads; every thread gets the result.  `scratch` holds NWAVES floats.  What a thread has stored
// to memory before is not waited for (the norms store the rows between their sums).
template <int NWAVES> __device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  if (NWAVES == 1) return v;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  lds_barrier();
  if (lane == 0) scratch[wave] = v;
  lds_barrier();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < NWAVES; ++i) t += scratch[i];
  return t;
}

template <int NWAVES> __device__ __forceinline__ float block_max(float v, float* scratch) {
  v = wave_max(v);
  if (NWAVES == 1) return v;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = scratch[0];
#pragma unroll
  for (int i = 1; i < NWAVES; ++i) t = fmaxf(t, scratch[i]);
  return t;
}

// Element type codes of the C interface.
enum DType : int { kF32 = 0, kBF16 = 1 };

// Four neighbouring values of a row as they come from memory (aligned to all four).  They become floats where they are used: a conversion
// beside the load would make the wave wait for it before it asks for the next.
template <typename T> struct Raw4 { float4 v; };
template <> struct Raw4<bf16_t> { uint2 v; };
__device__ __forceinline__ Raw4<float> fetch4(const float* p) { return {*reinterpret_cast<const float4*>(p)}; }
__device__ __forceinline__ Raw4<bf16_t> fetch4(const bf16_t* p) { return {*reinterpret_cast<const uint2*>(p)}; }
__device__ __forceinline__ float value4(const Raw4<float>& r, int i) { return i == 0 ? r.v.x : i == 1 ? r.v.y : i == 2 ? r.v.z : r.v.w; }
__device__ __forceinline__ float value4(const Raw4<bf16_t>& r, int i) {
  const uint32_t two = i < 2 ? r.v.x : r.v.y;
  return __uint_as_float(i & 1 ? two & 0xffff0000u : two << 16);
}

// sum[j] += the sum over `planes` planes, in the order of their index, of the four values at column 4 * col[j] of p.  The loads of up to
// PB planes are issued together (each is a trip to memory), in whole batches of PB, 4, 2 and 1: no load and no sum stands under a
// condition, which the compiler would take the loads along to, one by one (64 rows of 2,048 with eight planes and their norm 6.4 us then,
// 4.6 so).
template <int PB, int MAXJ, typename T, typename V>
__device__ __forceinline__ void add_some_planes(V (&sum)[MAXJ], const T* __restrict__ p, size_t stride, const int (&col)[MAXJ]) {
  Raw4<T> d[PB][MAXJ];
#pragma unroll
  for (int q = 0; q < PB; ++q)
#pragma unroll
    for (int j = 0; j < MAXJ; ++j) d[q][j] = fetch4(p + q * stride + 4 * col[j]);
#pragma unroll
  for (int q = 0; q < PB; ++q)
#pragma unroll
    for (int j = 0; j < MAXJ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[j].v[i] += value4(d[q][j], i);
}
template <int PB, int MAXJ, typename T, typename V>
__device__ __forceinline__ void add_planes(V (&sum)[MAXJ], const T* __restrict__ p, size_t stride, int planes, const int (&col)[MAXJ]) {
  static_assert(PB == 4 || PB == 8, "the batches of what is left are 4, 2 and 1");
  for (; planes >= PB; planes -= PB, p += PB * stride) add_some_planes<PB, MAXJ>(sum, p, stride, col);
  if (PB > 4 && planes & 4) add_some_planes<4, MAXJ>(sum, p, stride, col), p += 4 * stride;
  if (planes & 2) add_some_planes<2, MAXJ>(sum, p, stride, col), p += 2 * stride;
  if (planes & 1) add_some_planes<1, MAXJ>(sum, p, stride, col);
}

// One token of a causal convolution over time whose earlier inputs lie in the rows of `rows` (keep of them, `channels` apart), the
// last tap on `in`: added to y in the order of the taps.  x: the rows' values where there are at most four, which push_inputs then
// moves down by one row.
__device__ __forceinline__ float convolve_one(const float* rows, const float* __restrict__ taps, int keep, int channels, float in, float y,
                                              float (&x)[4]) {
  if (keep == 0) return fmaf(taps[0], in, y);
  if (keep <= 4) {                        // (in one stretch: one trip to memory)
    float w[4];
    const float last = taps[keep];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int at = min(j, keep - 1);
      x[j] = rows[at * channels];
      w[j] = taps[at];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) y = j < keep ? fmaf(w[j], x[j], y) : y;
    return fmaf(last, in, y);
  }
  for (int j = 0; j < keep; ++j) y = fmaf(taps[j], rows[(size_t)j * channels], y);
  return fmaf(taps[keep], in, y);
}
__device__ __forceinline__ void push_inputs(float* rows, int keep, int channels, float in, const float (&x)[4], bool held) {
  if (keep <= 0) return;
  if (held && keep <= 4) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
      if (r + 1 < keep) rows[(size_t)r * channels] = x[r + 1];
  } else {      // (ascending, so that a row is read before it is overwritten)
    for (int r = 0; r + 1 < keep; ++r) rows[(size_t)r * channels] = rows[(size_t)(r + 1) * channels];
  }
  rows[(size_t)(keep - 1) * channels] = in;
}

}  // namespace atoma

// Error codes of the C interface beyond hipError_t values (which are positive): negative numbers.
#define ATOMA_ERR_DTYPE (-2)
#define ATOMA_ERR_SHAPE (-3)

#define ATOMA_LAUNCH_CHECK()                     \
  do {                                           \
    hipError_t e__ = hipGetLastError();          \
    if (e__ != hipSuccess) return (int)e__;      \
  } while (0)
