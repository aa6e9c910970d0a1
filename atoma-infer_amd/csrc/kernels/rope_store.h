// The end of a fused q, k, v product: rotary encoding of its float32 sums and the write into the paged cache.
#pragma once
#include "cache_layout.h"
#include "common.h"

namespace atoma {

// What the rotary epilogue needs beside the product: see rope_store4.
struct RopeArgs {
  const int32_t* positions;      // [M]
  const float* cos_t;            // [positions, hd / 2]
  const float* sin_t;
  uint16_t* kcache;              // [pages, nkv, page_size * hd] tiles, bfloat16
  uint16_t* vcache;
  const int32_t* slot_mapping;   // [M]; negative: no cache write for the row
  int page_size, nh, nkv, hd;
};

// Outputs n0 .. n0 + 3 of row `row` of the fused q, k, v projection (float32 sums x0 .. x3), with the rows of every q
// and k head ordered so that the members of rotary pair i = (column i, column i + hd/2) are outputs 2i and 2i + 1 of
// the head: the four are two whole pairs, i and i + 1.  They are rotated here and go to their own columns: q to
// q_out [M, nh * hd], k into the row's slot of the paged cache (the order inside a tile: cache_layout.h); v heads are
// copied into theirs.  The same arithmetic as the rotary kernel (csrc/kernels/rotary.h:116-131 of the reference), on
// the float32 sums before they are rounded.
__device__ __forceinline__ void rope_store4(float x0, float x1, float x2, float x3, int row, int n0, const RopeArgs& ra,
                                            uint16_t* __restrict__ q_out, int ldq) {
  const int hd = ra.hd, half = hd >> 1;
  const int head = n0 / hd, d0 = n0 % hd;
  if (head >= ra.nh + ra.nkv) {
    const int slot = ra.slot_mapping[row];
    if (slot < 0) return;
    const int page = slot / ra.page_size, off = slot % ra.page_size;
    uint16_t* tile = ra.vcache + ((size_t)page * ra.nkv + (head - ra.nh - ra.nkv)) * ra.page_size * hd;
    tile[value_offset(d0, off, hd, ra.page_size)] = f32_to_bf16_bits(x0);
    tile[value_offset(d0 + 1, off, hd, ra.page_size)] = f32_to_bf16_bits(x1);
    tile[value_offset(d0 + 2, off, hd, ra.page_size)] = f32_to_bf16_bits(x2);
    tile[value_offset(d0 + 3, off, hd, ra.page_size)] = f32_to_bf16_bits(x3);
    return;
  }
  const int i = d0 >> 1;                       // even: columns i, i + 1 and their partners lie together
  const size_t at = (size_t)ra.positions[row] * half + i;
  const float c0 = ra.cos_t[at], s0 = ra.sin_t[at], c1 = ra.cos_t[at + 1], s1 = ra.sin_t[at + 1];
  const uint32_t lo = (uint32_t)f32_to_bf16_bits(x0 * c0 - x1 * s0) |
                      ((uint32_t)f32_to_bf16_bits(x2 * c1 - x3 * s1) << 16);      // columns i, i + 1
  const uint32_t hi = (uint32_t)f32_to_bf16_bits(x1 * c0 + x0 * s0) |
                      ((uint32_t)f32_to_bf16_bits(x3 * c1 + x2 * s1) << 16);      // i + half, i + half + 1
  if (head < ra.nh) {
    uint16_t* q = q_out + (size_t)row * ldq + (size_t)head * hd;
    *reinterpret_cast<uint32_t*>(q + i) = lo;
    *reinterpret_cast<uint32_t*>(q + i + half) = hi;
    return;
  }
  const int slot = ra.slot_mapping[row];
  if (slot < 0) return;
  const int page = slot / ra.page_size, off = slot % ra.page_size;
  uint16_t* tile = ra.kcache + ((size_t)page * ra.nkv + (head - ra.nh)) * ra.page_size * hd;
  *reinterpret_cast<uint32_t*>(tile + key_offset(off, i, ra.page_size)) = lo;
  *reinterpret_cast<uint32_t*>(tile + key_offset(off, i + half, ra.page_size)) = hi;
}

}  // namespace atoma
