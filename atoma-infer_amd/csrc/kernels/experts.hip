// Feed-forward layers that route every token to a few of many experts.
//
//   route_topk    per token: scores = sigmoid(router logits), or their softmax over all experts, in float32; the `top`
//                 experts with the largest score + correction[expert] (no correction: the score alone; the lower
//                 index wins a tie) with their weights, score * scale (the correction chooses, it does not weigh),
//                 or the experts with the largest logits, weighed by the softmax over the chosen logits alone (times
//                 scale); logits may have a bias per expert.  With groups (equal runs of neighbouring experts) a group's
//                 score is that of its best expert, and only experts of the best groups_keep groups can be chosen;
//                 A (token, choice) pair is a "slot", numbered token * top + choice;
//   route_group   one workgroup: slots ordered by expert (perm), where each expert's slots start (offsets), and the
//                 list of row tiles (expert, first place in perm) that the products below walk.  Which place a slot
//                 gets inside its expert's range is not fixed; no result depends on it, since every row of a product
//                 is computed by itself;
//   route_few     both in one launch, for few tokens of up to 64 experts;
//   expert_gemm   C[row(slot)] = (scale[slot] * A[src(slot)]) . W[expert]^T for all slots, tile by tile: true float32
//                 multiply-adds (gemm_f32_tile.h) over float32 or bfloat16 operands, every row's sums in the same
//                 order, so a row's result does not depend on the batch around it.  src is the slot's token (first product: the token's input, times its
//                 score) or the slot itself (second product); the second product writes choice c of token t to row
//                 c * T + t, so that the choices of a token lie in planes which the next norm adds in order.
//                 act = 2 squares what is positive of a result and drops the rest (experts without a gate: relu^2);
//                 out_scale[slot] multiplies a result (experts whose weight applies to their output).
#include "gate_act.h"
#include "gemm_f32_tile.h"

using namespace atoma;

constexpr int kTileM = 64, kTileN = 64;

// Up to 64 experts: lane e holds expert e and counts the experts that go before it (a larger score, or the same and a
// lower index), which is its place; the scores of the others come through scalar registers, one after the other, and no
// step waits for the one before.  The place of lane e's expert among the choices of the wave's token (top or more: not
// chosen), and its weight in `wt`.
__device__ __forceinline__ int rank_expert(const float* __restrict__ row, int experts, int top, int score,
                                           const float* __restrict__ correction, const float* __restrict__ bias,
                                           int groups, int groups_keep, float& wt) {
  const int e = threadIdx.x & 63;
  const bool real = e < experts;
  wt = real ? row[e] + (bias != nullptr ? bias[e] : 0.f) : -INFINITY;
  if (score == 1) {
    const float mx = wave_max(wt);
    wt = real ? expf(wt - mx) : 0.f;
    wt /= wave_sum(wt);
  } else if (score == 0) {
    wt = 1.0f / (1.0f + expf(-wt));
  }
  float sc = real ? (correction != nullptr ? wt + correction[e] : wt) : -INFINITY;
  if (!(sc == sc)) sc = -INFINITY;        // (scores that are no numbers come last: places stay a permutation)
  auto of = [](float v, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); };
  if (groups > 0) {
    const int size = experts / groups, mine = e / size;
    float best = -INFINITY;               // of this expert's group
    for (int g = 0; g < groups; ++g)
      for (int i = 0; i < size; ++i) {
        const float v = of(sc, g * size + i);
        best = fmaxf(best, mine == g ? v : -INFINITY);
      }
    int before = 0;
    for (int g = 0; g < groups; ++g) {
      const float v = of(best, g * size);
      before += v > best || (v == best && g < mine);
    }
    if (before >= groups_keep) sc = -INFINITY;
  }
  int place = 0;
  for (int i = 0; i < experts; ++i) {
    const float v = of(sc, i);
    place += v > sc || (v == sc && i < e);
  }
  if (!real) place = top;
  if (score == 2) {
    const bool chosen = place < top;
    const float mx = wave_max(chosen ? wt : -INFINITY);
    wt = chosen ? expf(wt - mx) : 0.f;
    wt /= wave_sum(wt);
  }
  return place;
}

__global__ void __launch_bounds__(256)
route_rank_kernel(const float* __restrict__ logits, int ld, int experts, int top, int32_t* __restrict__ ids,
                  float* __restrict__ weights, int n_tokens, int score, const float* __restrict__ correction,
                  float scale, const float* __restrict__ bias, int groups, int groups_keep) {
  const int e = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (t >= n_tokens) return;
  float wt;
  const int place = rank_expert(logits + (size_t)t * ld, experts, top, score, correction, bias, groups, groups_keep, wt);
  if (place < top) {
    ids[(size_t)t * top + place] = e;
    weights[(size_t)t * top + place] = wt * scale;
  }
}

// route_topk and route_group of few tokens in one launch: each kernel is a few hundred instructions behind a launch and
// a round trip to memory.  One workgroup; a wave ranks the experts of its token and takes a number at the counter of each
// chosen expert, which is the slot's place among that expert's.  Behind one barrier lane e of every wave holds expert e's
// count, and a scan over the lanes gives where each expert's slots and tiles start.  Two launches / this one in a graph, us,
// 1 / 8 / 16 tokens: 8 of 8 experts 3.7 / 4.4 / 4.7 -> 2.8 / 2.8 / 3.1, 4 of 32 5.6 / 6.8 / 7.2 -> 3.9 / 3.9 / 4.6, 6 of 64 in
// eight groups 11.2 / 12.9 / 13.8 -> 7.9 / 8.3 / 10.7.  No more than a token a wave: with two in turn the last of these takes
// 19.4 against 14.0, with four the second 11.2 against 7.6.
constexpr int kRouteFew = 16;        // tokens, a wave each

__global__ void __launch_bounds__(kRouteFew * 64)
route_few_kernel(const float* __restrict__ logits, int ld, int experts, int top, int32_t* __restrict__ ids,
                 float* __restrict__ weights, int n_tokens, int score, const float* __restrict__ correction,
                 float scale, const float* __restrict__ bias, int groups, int groups_keep, int32_t* __restrict__ perm,
                 int32_t* __restrict__ offsets, int32_t* __restrict__ tiles, int max_tiles, int tile_m) {
  __shared__ int32_t counts[64];
  const int e = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x < 64) counts[threadIdx.x] = 0;
  __syncthreads();
  int slot = -1, number = 0;
  if (wave < n_tokens) {
    float wt;
    const int place = rank_expert(logits + (size_t)wave * ld, experts, top, score, correction, bias, groups, groups_keep, wt);
    if (place < top) {
      slot = wave * top + place;
      number = atomicAdd(&counts[e], 1);
      ids[slot] = e;
      weights[slot] = wt * scale;
    }
  }
  __syncthreads();
  const int count = counts[e], mine = (count + tile_m - 1) / tile_m;
  int at = count, tile = mine;         // inclusive sums over the lanes, then exclusive ones
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int a = __shfl_up(at, off, 64), b = __shfl_up(tile, off, 64);
    if (e >= off) at += a, tile += b;
  }
  const int all = __shfl(tile, 63, 64);
  at -= count, tile -= mine;
  if (slot >= 0) perm[at + number] = slot;
  if (wave == 0) {
    if (e < experts) offsets[e] = at;
    if (e == experts - 1) offsets[experts] = at + count;
    for (int i = 0; i < mine; ++i) tiles[2 * (tile + i)] = e, tiles[2 * (tile + i) + 1] = at + i * tile_m;
    for (int i = all + e; i < max_tiles; i += 64) tiles[2 * i] = -1, tiles[2 * i + 1] = 0;
  }
}

template <bool GROUPED>
__global__ void __launch_bounds__(256)
route_topk_kernel(const float* __restrict__ logits, int ld, int experts, int top, int32_t* __restrict__ ids,
                  float* __restrict__ weights, int n_tokens, int score, const float* __restrict__ correction,
                  float scale, const float* __restrict__ bias, int groups, int groups_keep) {
  // a wave a token; lane l holds experts l, l + 64, ...
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (!GROUPED && row >= n_tokens) return;
  // (with groups all waves meet at barriers: one without a token works on the last one and stores nothing)
  const int t = row < n_tokens ? row : n_tokens - 1;
  constexpr int PER = 16;      // experts <= 1024
  // sc: what chooses (score, plus the correction where there is one); wt: what weighs (the score alone)
  // score 0: sigmoid; 1: softmax over all experts; 2: the logits choose, softmax over the chosen ones (below)
  float sc[PER], wt[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + j * 64;
    wt[j] = e < experts ? logits[(size_t)t * ld + e] + (bias != nullptr ? bias[e] : 0.f) : -INFINITY;
  }
  if (score == 1) {
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER; ++j) mx = fmaxf(mx, wt[j]);
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      wt[j] = lane + j * 64 < experts ? expf(wt[j] - mx) : 0.f;
      sum += wt[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PER; ++j) wt[j] /= sum;
  } else if (score == 0) {
#pragma unroll
    for (int j = 0; j < PER; ++j) wt[j] = lane + j * 64 < experts ? 1.0f / (1.0f + expf(-wt[j])) : 0.f;
  }
  float first = 0.f, total = 0.f, mine = 0.f;      // score 2: the largest logit, the sum, and lane c's choice c
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = lane + j * 64;
    sc[j] = e < experts ? (correction != nullptr ? wt[j] + correction[e] : wt[j]) : -INFINITY;
  }
  if constexpr (GROUPED) {
    // the scores of a wave's token in LDS, then its groups' scores over them; lane l holds groups l, l + 64, ...
    __shared__ float table[4][1024];
    float* const mine_t = table[threadIdx.x >> 6];
    const int size = experts / groups;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + j * 64 < experts) mine_t[lane + j * 64] = sc[j];
    __syncthreads();
    float gs[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      gs[j] = -INFINITY;
      const int g = lane + j * 64;
      if (g < groups)
        for (int e = 0; e < size; ++e) gs[j] = fmaxf(gs[j], mine_t[g * size + e]);
    }
    __syncthreads();
    // a kept group is marked where its scores were
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + j * 64 < groups) mine_t[lane + j * 64] = 0.f;
    for (int c = 0; c < groups_keep; ++c) {
      float best = -INFINITY;
      int arg = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (gs[j] > best) best = gs[j], arg = lane + j * 64;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, 64);
        const int oa = __shfl_xor(arg, off, 64);
        if (ob > best || (ob == best && oa < arg)) best = ob, arg = oa;
      }
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if (lane + j * 64 == arg) {
          gs[j] = -INFINITY;
          mine_t[arg] = 1.f;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + j * 64 < experts && mine_t[(lane + j * 64) / size] == 0.f) sc[j] = -INFINITY;
    if (row >= n_tokens) return;
  }
  for (int c = 0; c < top; ++c) {
    float best = -INFINITY, bw = 0.f;
    int arg = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (sc[j] > best) best = sc[j], bw = wt[j], arg = lane + j * 64;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const float ow = __shfl_xor(bw, off, 64);
      const int oa = __shfl_xor(arg, off, 64);
      if (ob > best || (ob == best && oa < arg)) best = ob, bw = ow, arg = oa;
    }
    if (arg >= experts) arg = c, bw = 0.f;     // logits that are no numbers: still an expert of the layer
    if (score == 2) {
      if (c == 0) first = bw;
      bw = expf(bw - first);
      total += bw;
      // weights of a choice wait for the sum: 64 choices a round in the wave's lanes, more through memory
      if (top <= 64) { if (lane == c) mine = bw; }
      else if (lane == 0) weights[(size_t)t * top + c] = bw;
    } else if (lane == 0) {
      weights[(size_t)t * top + c] = bw * scale;
    }
    if (lane == 0) ids[(size_t)t * top + c] = arg;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (lane + j * 64 == arg) sc[j] = -INFINITY;
  }
  if (score == 2) {
    if (top <= 64) { if (lane < top) weights[(size_t)t * top + lane] = mine / total * scale; }
    else if (lane == 0) { for (int c = 0; c < top; ++c) weights[(size_t)t * top + c] *= scale / total; }
  }
}

__global__ void __launch_bounds__(1024)
route_group_kernel(const int32_t* __restrict__ ids, int n_slots, int experts, int32_t* __restrict__ perm,
                   int32_t* __restrict__ offsets, int32_t* __restrict__ tiles, int max_tiles, int tile_m) {
  __shared__ int32_t counts[1024];
  __shared__ int32_t cursor[1024];
  for (int e = threadIdx.x; e < experts; e += 1024) counts[e] = 0;
  __syncthreads();
  for (int s = threadIdx.x; s < n_slots; s += 1024) atomicAdd(&counts[ids[s]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, n = 0;
    for (int e = 0; e < experts; ++e) {
      offsets[e] = at;
      cursor[e] = at;
      for (int r = 0; r < counts[e]; r += tile_m) {
        tiles[2 * n] = e;
        tiles[2 * n + 1] = at + r;
        ++n;
      }
      at += counts[e];
    }
    offsets[experts] = at;
    for (; n < max_tiles; ++n) tiles[2 * n] = -1, tiles[2 * n + 1] = 0;
  }
  __syncthreads();
  for (int s = threadIdx.x; s < n_slots; s += 1024) perm[atomicAdd(&cursor[ids[s]], 1)] = s;
}

template <bool VEC, typename TA, typename TW, typename TC>
__global__ void __launch_bounds__(256)
expert_gemm_kernel(const TA* __restrict__ a, int lda, int a_div, const float* __restrict__ scale,
                   const TW* __restrict__ w, TC* __restrict__ c, int ldc, int N, int K,
                   const int32_t* __restrict__ perm, const int32_t* __restrict__ offsets,
                   const int32_t* __restrict__ tiles, int top, int plane_rows, int act,
                   const float* __restrict__ out_scale) {
  __shared__ __attribute__((aligned(16))) float lds[2 * (kTileM + kTileN) * kF32Row];
  const int e = tiles[2 * blockIdx.y];
  if (e < 0) return;
  const int row0 = tiles[2 * blockIdx.y + 1], row_end = offsets[e + 1];
  const int n0 = blockIdx.x * kTileN;
  const TW* we = w + (size_t)e * N * K;
  auto slot_of = [&](int r) { return row0 + r < row_end ? perm[row0 + r] : -1; };
  f32x4_t acc[kTileN / 32][kTileM / 32];
  f32_tile<kTileM, kTileN, VEC, false, TA, TW>(
      lds, K, 0,
      [&](int r) { return a + (size_t)(perm[min(row0 + r, row_end - 1)] / a_div) * lda; },
      [&](int r) { return we + (size_t)min(n0 + r, N - 1) * K; },
      [&](int r) { return scale != nullptr ? scale[perm[min(row0 + r, row_end - 1)]] : 1.f; }, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < kTileM / 32; ++j) {
    const int slot = slot_of((wave >> 1) * (kTileM / 2) + j * 16 + (lane & 15));
    if (slot < 0) continue;
    const size_t row = plane_rows > 0 ? (size_t)(slot % top) * plane_rows + slot / top : (size_t)slot;
    const float os = out_scale != nullptr ? out_scale[slot] : 1.0f;
#pragma unroll
    for (int i = 0; i < kTileN / 32; ++i)
#pragma unroll
      for (int l = 0; l < 4; ++l) {
        const int n = n0 + (wave & 1) * (kTileN / 2) + i * 16 + (lane >> 4) * 4 + l;
        float v = acc[i][j][l];
        if (act == 2) v = v > 0.f ? v * v : 0.f;
        if (n < N) c[row * ldc + n] = from_f32<TC>(v * os);
      }
  }
}

// ---- bfloat16 on the matrix cores -------------------------------------------------------------------------------
//
//   gather_scale      xs[place] = bfloat16(score[slot] * x[token of slot]) for every place of perm: the inputs of the
//                     first product, ordered by expert, so that a tile's rows are contiguous;
//   expert_gemm_mfma  a workgroup takes a tile of up to 64 places of one expert against 128 rows of that expert's
//                     weight, v_mfma_f32_16x16x32_bf16 with float32 sums: the weight's fragments come straight from
//                     global memory (an element is used by one wave only), the tile of activations passes LDS, 64
//                     columns of K at a time, and is shared by the four waves; both are asked for a step ahead.  Tiles
//                     hold 64 places, or 128 where the experts have many (prompts); blocks of 16 places without a live
//                     one are skipped.  It serves what the streaming kernel below (few places an expert) and the dense
//                     products' tile kernel (SiLU, many places) do not take: other gates and relu^2 with many places,
//                     runs of 20 to 30 places that leave those tiles barely filled, and widths that are no multiple of
//                     64 or 128.  SWIGLU: the weight's rows come in blocks of 16 gate rows followed by the 16 up
//                     rows of the same outputs, a lane then holds a gate value and its up value, and silu(gate) * up
//                     leaves as bfloat16 [places, ff]; else the float32 result goes to the plane and row of the
//                     place's slot (choice c of token t: row c * T + t).
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__global__ void __launch_bounds__(256)
gather_scale_kernel(const uint16_t* __restrict__ x, int ldx, const float* __restrict__ score,
                    const int32_t* __restrict__ perm, uint16_t* __restrict__ xs, int K, int top) {
  const int place = blockIdx.x, slot = perm[place];
  const float sc = score != nullptr ? score[slot] : 1.0f;      // (no scores: the inputs as they are)
  const uint16_t* src = x + (size_t)(slot / top) * ldx;
  for (int k = threadIdx.x; k < K; k += 256) xs[(size_t)place * K + k] = f32_to_bf16_bits(bf16_bits_to_f32(src[k]) * sc);
}


// NS: blocks of 16 rows of the weight a wave takes.  KSUB: pieces of 32 columns of K a step (2, or 4 for tiles of 64
// places, which hold few: the product then streams the weight, and what it needs is many bytes in flight a step).
// ACT: 0 the float32 result (times out_scale[slot] where given) by place or by slot; 1 silu(gate) * up, or a relative
// of it (gate_act.h), over interleaved rows, bfloat16 [places, N / 2]; 2 relu^2 of the result, bfloat16 [places, N].
template <int ACT, int TM, int NS, int KSUB>
__global__ void __launch_bounds__(256)
expert_gemm_mfma_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, void* __restrict__ c, int ldc,
                        int N, int K, const int32_t* __restrict__ perm, const int32_t* __restrict__ offsets,
                        const int32_t* __restrict__ tiles, int top, int plane_rows,
                        const float* __restrict__ out_scale, GateAct gate) {
  constexpr bool SWIGLU = ACT == 1;
  constexpr int MS = TM / 16;          // blocks of 16 places a tile
  constexpr int KSTEP = 32 * KSUB;     // columns of K a step
  constexpr int kLdsRow = KSTEP + 8;   // bfloat16 elements a row of the activations' tile takes in LDS (padded)
  constexpr int SEGS = KSTEP / 8;      // 16-byte pieces a row of the tile
  constexpr int AP = TM * SEGS / 256;  // ... and a thread moves a step
  __shared__ __attribute__((aligned(16))) uint16_t at[TM * kLdsRow];
  const int e = tiles[2 * blockIdx.y];
  if (e < 0) return;
  const int row0 = tiles[2 * blockIdx.y + 1];
  const int rows = min(TM, offsets[e + 1] - row0);
  const int msub = (rows + 15) >> 4;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n_base = blockIdx.x * (64 * NS) + wave * (16 * NS);
  // (a wave whose columns lie beyond N still joins the barriers below; its rows are clamped and never stored)
  const uint16_t* we = w + (size_t)e * N * K;
  const uint16_t* wp[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    int n = n_base + s * 16 + r16;
    if (n > N - 1) n = N - 1;
    wp[s] = we + (size_t)n * K + kg * 8;
  }
  f32x4 acc[NS][MS];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int m = 0; m < MS; ++m) acc[s][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The operands of a step are asked for a step ahead: the weight's fragments wait in registers, the activations' pieces
  // too, until the tile of the step before has been read and they may go to LDS.
  bf16x8 wf[KSUB][NS], wn[KSUB][NS];
  uint4 ar[AP];
  auto fetch = [&](int k0, bf16x8 (&dst)[KSUB][NS]) {
#pragma unroll
    for (int kk = 0; kk < KSUB; ++kk)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        // (K is a multiple of 32: the last step may be short)
        if (k0 + kk * 32 < K) dst[kk][s] = *reinterpret_cast<const bf16x8*>(wp[s] + k0 + kk * 32);
        else dst[kk][s] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      }
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      const int idx = tid + i * 256, r = idx / SEGS, seg = idx % SEGS;
      ar[i] = make_uint4(0, 0, 0, 0);
      if (r < rows && k0 + seg * 8 < K) ar[i] = *reinterpret_cast<const uint4*>(a + (size_t)(row0 + r) * K + k0 + seg * 8);
    }
  };
  fetch(0, wf);
  for (int k0 = 0; k0 < K; k0 += KSTEP) {
    __syncthreads();          // the tile of the step before has been read
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      const int idx = tid + i * 256, r = idx / SEGS, seg = idx % SEGS;
      if (r < msub * 16) *reinterpret_cast<uint4*>(at + r * kLdsRow + seg * 8) = ar[i];
    }
    __syncthreads();
    if (k0 + KSTEP < K) fetch(k0 + KSTEP, wn);
#pragma unroll
    for (int kk = 0; kk < KSUB; ++kk) {
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        if (m < msub) {
          const bf16x8 af = *reinterpret_cast<const bf16x8*>(at + (m * 16 + r16) * kLdsRow + kk * 32 + kg * 8);
#pragma unroll
          for (int s = 0; s < NS; ++s)
            acc[s][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kk][s], af, acc[s][m], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int kk = 0; kk < KSUB; ++kk)
#pragma unroll
      for (int s = 0; s < NS; ++s) wf[kk][s] = wn[kk][s];
  }
  // lane: place m * 16 + r16 of the tile, columns kg * 4 .. + 3 of each of its NS blocks of 16 rows of the weight
#pragma unroll
  for (int m = 0; m < MS; ++m) {
    const int r = m * 16 + r16;
    if (m >= msub || r >= rows) continue;
    const int place = row0 + r;
    if constexpr (SWIGLU) {
#pragma unroll
      for (int s = 0; s < NS; s += 2) {        // blocks come in pairs: 16 gate rows, then their 16 up rows
        const int n0 = (n_base + s * 16) / 2 + kg * 4;      // outputs: one for every pair of a gate row and an up row
        uint16_t* dst = (uint16_t*)c + (size_t)place * ldc + n0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (n_base + s * 16 + 16 + kg * 4 + i < N)
            dst[i] = f32_to_bf16_bits(gated(acc[s][m][i], acc[s + 1][m][i], gate));
        }
      }
    } else if constexpr (ACT == 2) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int n0 = n_base + s * 16 + kg * 4;
        uint16_t* dst = (uint16_t*)c + (size_t)place * ldc + n0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float v = acc[s][m][i];
          if (n0 + i < N) dst[i] = f32_to_bf16_bits(v > 0.f ? v * v : 0.f);
        }
      }
    } else {
      const int slot = perm[place];
      const size_t row = plane_rows > 0 ? (size_t)(slot % top) * plane_rows + slot / top : (size_t)place;
      const float os = out_scale != nullptr ? out_scale[slot] : 1.0f;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int n0 = n_base + s * 16 + kg * 4;
        float* dst = (float*)c + row * ldc + n0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n0 + i < N) dst[i] = acc[s][m][i] * os;
      }
    }
  }
}

// Few places an expert (decode steps): the product only streams the chosen experts' weights, and what bounds it is the bytes
// in flight.  A workgroup takes 32 rows of an expert's weight against a tile of up to 16 places; its four waves split K,
// fetch both operands straight from memory, two batches of four steps in turn, and meet in LDS.  With the scores given
// (scale) the inputs are the tokens' rows themselves, scaled and rounded as gather_scale does it, so that no kernel has
// to lay them out before.  8 experts of 1,024 columns at width 2,048, 8 places each, with the grouping: 25 us, where the
// tiles of 64 places (128 columns of K a step, one step ahead: 34 + 18 us alone) and gather_scale took 50.
constexpr int kStreamPlaces = 16, kStreamWaves = 4;

template <int ACT, bool GATHER, bool SCALED>
__global__ void __launch_bounds__(64 * kStreamWaves)
expert_stream_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, const int32_t* __restrict__ tiles,
                     const int32_t* __restrict__ offsets, const int32_t* __restrict__ perm, int K, int N, int lda, int top,
                     const float* __restrict__ scale, void* __restrict__ c, int ldc, int plane_rows,
                     const float* __restrict__ out_scale, GateAct gate) {
  constexpr int U = 4;
  __shared__ f32x4 red[kStreamWaves - 1][2][64];
  const int e = tiles[2 * blockIdx.y];
  if (e < 0) return;
  const int row0 = tiles[2 * blockIdx.y + 1], rows = min(kStreamPlaces, offsets[e + 1] - row0);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 32, k_len = K / kStreamWaves, k_begin = wave * k_len;
  const int place = row0 + min(r16, rows - 1), slot = perm[place];      // (rows past the tile: its last, never stored)
  const uint16_t* const ap = a + (size_t)(GATHER ? slot / top : place) * lda + k_begin + kg * 8;
  const float sc = SCALED ? scale[slot] : 1.f;
  const uint16_t* const wp = w + ((size_t)e * N + n0 + r16) * K + k_begin + kg * 8;
  const size_t block = (size_t)16 * K;
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  bf16x8 wf[2][U][2], af[2][U];
  auto load = [&](int buf, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int s = 0; s < 2; ++s) wf[buf][u][s] = *reinterpret_cast<const bf16x8*>(wp + s * block + k0 + u * 32);
      af[buf][u] = *reinterpret_cast<const bf16x8*>(ap + k0 + u * 32);
    }
  };
  auto one = [&](bf16x8 x, const bf16x8 (&y)[2]) {
    if constexpr (SCALED) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (__bf16)((float)x[i] * sc);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y[s], x, acc[s], 0, 0, 0);
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u) one(af[buf][u], wf[buf][u]);
  };
  const int batches = k_len / (32 * U);
  if (batches > 0) load(0, 0);
  int b = 0;
  for (; b + 2 <= batches; b += 2) {
    load(1, (b + 1) * 32 * U);
    multiply(0);
    if (b + 2 < batches) load(0, (b + 2) * 32 * U);
    multiply(1);
  }
  if (b < batches) multiply(0);
  for (int k = batches * 32 * U; k < k_len; k += 32) {
    bf16x8 y[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) y[s] = *reinterpret_cast<const bf16x8*>(wp + s * block + k);
    one(*reinterpret_cast<const bf16x8*>(ap + k), y);
  }
  if (wave > 0) {
#pragma unroll
    for (int s = 0; s < 2; ++s) red[wave - 1][s][lane] = acc[s];
  }
  __syncthreads();
  if (wave > 0 || r16 >= rows) return;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < kStreamWaves - 1; ++i) acc[s] += red[i][s][lane];
  if constexpr (ACT == 1) {          // 16 gate rows, then the 16 up rows of the same outputs
    uint16_t* const dst = (uint16_t*)c + (size_t)place * ldc + n0 / 2 + kg * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i] = f32_to_bf16_bits(gated(acc[0][i], acc[1][i], gate));
  } else if constexpr (ACT == 2) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = acc[s][i];
        ((uint16_t*)c)[(size_t)place * ldc + n0 + s * 16 + kg * 4 + i] = f32_to_bf16_bits(v > 0.f ? v * v : 0.f);
      }
  } else {
    const size_t row = plane_rows > 0 ? (size_t)(slot % top) * plane_rows + slot / top : (size_t)place;
    const float os = out_scale != nullptr ? out_scale[slot] : 1.0f;
    float* const dst = (float*)c + row * ldc + n0 + kg * 4;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[s * 16 + i] = acc[s][i] * os;
  }
}

// out[t, i] = relu(u[t, i])^2 * sigmoid(u[t, off_gate]) for an expert that every token uses: its first product's
// result u [T, ld] holds the ff columns of the expert and, at off_gate, the token's gate (off_gate < 0: no gate).
template <typename TI, typename TO>
__global__ void __launch_bounds__(256)
relu2_gate_kernel(const TI* __restrict__ u, int ld, TO* __restrict__ out, int ff, int off_gate) {
  const size_t t = blockIdx.x;
  const float g = off_gate >= 0 ? 1.0f / (1.0f + expf(-to_f32(u[t * ld + off_gate]))) : 1.0f;
  for (int i = threadIdx.x; i < ff; i += 256) {
    const float v = to_f32(u[t * ld + i]);
    out[t * ff + i] = from_f32<TO>(v > 0.f ? v * v * g : 0.f);
  }
}

extern "C" int atoma_relu2_gate(const void* u, int u_dtype, int ld, void* out, int out_dtype, int n_tokens, int ff,
                                int off_gate, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (ff <= 0 || ld < ff || off_gate >= ld) return ATOMA_ERR_SHAPE;
  dim3 grid(n_tokens), block(256);
  if (u_dtype == kF32 && out_dtype == kF32)
    hipLaunchKernelGGL((relu2_gate_kernel<float, float>), grid, block, 0, stream, (const float*)u, ld, (float*)out, ff,
                       off_gate);
  else if (u_dtype == kF32 && out_dtype == kBF16)
    hipLaunchKernelGGL((relu2_gate_kernel<float, bf16_t>), grid, block, 0, stream, (const float*)u, ld, (bf16_t*)out,
                       ff, off_gate);
  else if (u_dtype == kBF16 && out_dtype == kBF16)
    hipLaunchKernelGGL((relu2_gate_kernel<bf16_t, bf16_t>), grid, block, 0, stream, (const bf16_t*)u, ld, (bf16_t*)out,
                       ff, off_gate);
  else
    return ATOMA_ERR_DTYPE;
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_gather_scale(const void* x, int ldx, const float* score, const int32_t* perm, void* xs, int K,
                                  int top, int n_slots, hipStream_t stream) {
  if (n_slots <= 0) return 0;
  if (K <= 0 || ldx < K || top <= 0) return ATOMA_ERR_SHAPE;
  hipLaunchKernelGGL(gather_scale_kernel, dim3(n_slots), dim3(256), 0, stream, (const uint16_t*)x, ldx, score, perm,
                     (uint16_t*)xs, K, top);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// a [places, K] bfloat16 in the order of perm; w [experts, N, K] bfloat16.  act 1: c bfloat16 [places, N / 2] (ldc),
// the rows of w in blocks of 16 gate rows and their 16 up rows; act 2: c bfloat16 [places, N], relu^2; act 0: c
// float32, by place or (plane_rows > 0) by slot, times out_scale[slot] where given
extern "C" int atoma_expert_gemm_mfma(const void* a, const void* w, void* c, int ldc, int N, int K, const int32_t* perm,
                                      const int32_t* offsets, const int32_t* tiles, int max_tiles, int top,
                                      int plane_rows, int act, int tile_m, const float* out_scale,
                                      int gate_kind, float limit, float slope, hipStream_t stream) {
  if (max_tiles <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 32 || N % 32 || (tile_m != 64 && tile_m != 128) || top <= 0 || max_tiles > 65535 || ((uintptr_t)a & 15) || ((uintptr_t)w & 15) ||
      act < 0 || act > 2 || !gate_act_ok(gate_kind, limit) || ldc < (act == 1 ? N / 2 : N) || (act != 0 && (plane_rows > 0 || out_scale != nullptr)))
    return ATOMA_ERR_SHAPE;
  const GateAct gate{gate_kind, limit, slope};
  const int ns = 2;      // (four blocks a wave measured slower for tiles of 128 places: 467 against 336 us)
  dim3 grid((N + 64 * ns - 1) / (64 * ns), max_tiles), block(256);
#define ATOMA_EGM(SW, TM_, NS_, KSUB_)                                                                           \
  hipLaunchKernelGGL((expert_gemm_mfma_kernel<SW, TM_, NS_, KSUB_>), grid, block, 0, stream, (const uint16_t*)a, \
                     (const uint16_t*)w, c, ldc, N, K, perm, offsets, tiles, top, plane_rows, out_scale, gate)
  if (act == 1 && tile_m == 64) ATOMA_EGM(1, 64, 2, 4);
  else if (act == 1) ATOMA_EGM(1, 128, 2, 2);
  else if (act == 2 && tile_m == 64) ATOMA_EGM(2, 64, 2, 4);
  else if (act == 2) ATOMA_EGM(2, 128, 2, 2);
  else if (tile_m == 64) ATOMA_EGM(0, 64, 2, 4);
  else ATOMA_EGM(0, 128, 2, 2);
#undef ATOMA_EGM
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// The product for few places an expert.  gather: a is [tokens, K] (row stride lda) and a place's input is its token's row,
// times scale[slot] where given; else a is [places, K].  tiles as route_group makes them for 16 places.
extern "C" int atoma_expert_stream(const void* a, int lda, int gather, const float* scale, const void* w, void* c, int ldc,
                                   int N, int K, const int32_t* perm, const int32_t* offsets, const int32_t* tiles,
                                   int max_tiles, int top, int plane_rows, int act, const float* out_scale, int gate_kind,
                                   float limit, float slope, hipStream_t stream) {
  if (max_tiles <= 0 || N <= 0) return 0;
  if (K <= 0 || K % (32 * kStreamWaves) || N % 32 || lda < K || lda % 8 || top <= 0 || max_tiles > 65535 || ((uintptr_t)a & 15) ||
      ((uintptr_t)w & 15) || act < 0 || act > 2 || !gate_act_ok(gate_kind, limit) || ldc < (act == 1 ? N / 2 : N) ||
      (act != 0 && (plane_rows > 0 || out_scale != nullptr)) || (scale != nullptr && !gather))
    return ATOMA_ERR_SHAPE;
  const GateAct gate{gate_kind, limit, slope};
  const dim3 grid(N / 32, max_tiles), block(64 * kStreamWaves);
#define ATOMA_ES(ACT, G, S)                                                                                            \
  hipLaunchKernelGGL((expert_stream_kernel<ACT, G, S>), grid, block, 0, stream, (const uint16_t*)a, (const uint16_t*)w, tiles, \
                     offsets, perm, K, N, lda, top, scale, c, ldc, plane_rows, out_scale, gate)
#define ATOMA_ES_(ACT)                          \
  do {                                          \
    if (scale != nullptr) ATOMA_ES(ACT, true, true); \
    else if (gather) ATOMA_ES(ACT, true, false); \
    else ATOMA_ES(ACT, false, false);           \
  } while (0)
  if (act == 1) ATOMA_ES_(1);
  else if (act == 2) ATOMA_ES_(2);
  else ATOMA_ES_(0);
#undef ATOMA_ES_
#undef ATOMA_ES
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_route_topk(const float* logits, int ld, int experts, int top, int32_t* ids, float* weights,
                                int n_tokens, int score, const float* correction, float scale, const float* bias,
                                int groups, int groups_keep, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (experts <= 0 || experts > 1024 || top <= 0 || top > experts || ld < experts || score < 0 ||
      score > 2)
    return ATOMA_ERR_SHAPE;
  // groups: 0 (none), or a number of equal runs of experts, of which groups_keep hold at least the top experts
  if (groups < 0 || (groups > 0 && (experts % groups || groups_keep <= 0 || groups_keep > groups ||
                                    groups_keep * (experts / groups) < top)))
    return ATOMA_ERR_SHAPE;
  const dim3 grid((n_tokens + 3) / 4), block(256);
  if (groups <= groups_keep) groups = groups_keep = 0;      // (all groups are kept)
  if (experts <= 64)
    hipLaunchKernelGGL(route_rank_kernel, grid, block, 0, stream, logits, ld, experts, top, ids, weights, n_tokens, score,
                       correction, scale, bias, groups, groups_keep);
  else if (groups > 0)
    hipLaunchKernelGGL(route_topk_kernel<true>, grid, block, 0, stream, logits, ld, experts, top, ids, weights, n_tokens,
                       score, correction, scale, bias, groups, groups_keep);
  else
    hipLaunchKernelGGL(route_topk_kernel<false>, grid, block, 0, stream, logits, ld, experts, top, ids, weights, n_tokens,
                       score, correction, scale, bias, 0, 0);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// the most row tiles of tile_m places that n_slots slots of `experts` experts can need
extern "C" int atoma_route_max_tiles(int n_slots, int experts, int tile_m) {
  const int full = n_slots / tile_m + experts;
  return full < n_slots ? full : (n_slots > 0 ? n_slots : 1);
}

// route_topk, then route_group with tiles of tile_m places, in one launch: up to 64 experts, up to 16 tokens
extern "C" int atoma_route_few(const float* logits, int ld, int experts, int top, int32_t* ids, float* weights,
                               int n_tokens, int score, const float* correction, float scale, const float* bias,
                               int groups, int groups_keep, int32_t* perm, int32_t* offsets, int32_t* tiles,
                               int max_tiles, int tile_m, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (n_tokens > kRouteFew || experts <= 0 || experts > 64 || top <= 0 || top > experts || ld < experts || score < 0 ||
      score > 2 || (tile_m != 16 && tile_m != 64 && tile_m != 128 && tile_m != 256) ||
      max_tiles < atoma_route_max_tiles(n_tokens * top, experts, tile_m))
    return ATOMA_ERR_SHAPE;
  if (groups < 0 || (groups > 0 && (experts % groups || groups_keep <= 0 || groups_keep > groups ||
                                    groups_keep * (experts / groups) < top)))
    return ATOMA_ERR_SHAPE;
  if (groups <= groups_keep) groups = groups_keep = 0;      // (all groups are kept)
  hipLaunchKernelGGL(route_few_kernel, dim3(1), dim3(kRouteFew * 64), 0, stream, logits, ld, experts, top, ids, weights,
                     n_tokens, score, correction, scale, bias, groups, groups_keep, perm, offsets, tiles, max_tiles,
                     tile_m);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_route_group(const int32_t* ids, int n_slots, int experts, int32_t* perm, int32_t* offsets,
                                 int32_t* tiles, int max_tiles, int tile_m, hipStream_t stream) {
  if (n_slots <= 0) return 0;
  if (experts <= 0 || experts > 1024 || (tile_m != 16 && tile_m != 64 && tile_m != 128 && tile_m != 256) ||
      max_tiles < atoma_route_max_tiles(n_slots, experts, tile_m))
    return ATOMA_ERR_SHAPE;
  hipLaunchKernelGGL(route_group_kernel, dim3(1), dim3(1024), 0, stream, ids, n_slots, experts, perm, offsets, tiles,
                     max_tiles, tile_m);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

extern "C" int atoma_expert_gemm(const void* a, int a_dtype, int lda, int a_div, const float* scale, const void* w,
                                 int w_dtype, void* c, int c_dtype, int ldc, int N, int K, const int32_t* perm,
                                 const int32_t* offsets, const int32_t* tiles, int max_tiles, int top, int plane_rows,
                                 int act, const float* out_scale, hipStream_t stream) {
  if (max_tiles <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N || a_div <= 0 || top <= 0 || max_tiles > 65535 || (act != 0 && act != 2))
    return ATOMA_ERR_SHAPE;
  dim3 grid((N + kTileN - 1) / kTileN, max_tiles), block(256);
#define ATOMA_EG_(V, TA, TW, TC)                                                                                   \
  hipLaunchKernelGGL((expert_gemm_kernel<V, TA, TW, TC>), grid, block, 0, stream, (const TA*)a, lda, a_div, scale, \
                     (const TW*)w, (TC*)c, ldc, N, K, perm, offsets, tiles, top, plane_rows, act, out_scale)
  // (pieces of four values: at most 16 bytes)
  const bool vec = K % kF32Step == 0 && lda % 4 == 0 && ((uintptr_t)a & 15) == 0 && ((uintptr_t)w & 15) == 0;
#define ATOMA_EG(TA, TW, TC)                \
  do {                                      \
    if (vec) ATOMA_EG_(true, TA, TW, TC);   \
    else ATOMA_EG_(false, TA, TW, TC);      \
  } while (0)
  if (a_dtype == kF32 && w_dtype == kF32 && c_dtype == kF32) ATOMA_EG(float, float, float);
  else if (a_dtype == kF32 && w_dtype == kBF16 && c_dtype == kF32) ATOMA_EG(float, bf16_t, float);
  else if (a_dtype == kBF16 && w_dtype == kBF16 && c_dtype == kF32) ATOMA_EG(bf16_t, bf16_t, float);
  else if (a_dtype == kBF16 && w_dtype == kBF16 && c_dtype == kBF16) ATOMA_EG(bf16_t, bf16_t, bf16_t);
  else return ATOMA_ERR_DTYPE;
#undef ATOMA_EG
#undef ATOMA_EG_
  ATOMA_LAUNCH_CHECK();
  return 0;
}
