// Paged attention for any head size up to 256 (multiples of 8), any page size, float32 or bfloat16: the general kernel.
// It serves the true 32-bit path and every shape that the bfloat16 MFMA kernels refuse.
//
// The token at absolute position p of request s attends keys [max(0, p - window + 1), p] of that request, read through
// its block table, after this step's keys and values have been written.  That one rule covers whole prompts, portions of
// prompts and single decoded tokens (bottom-right aligned causal mask, csrc/kernels/mask.h:171-172 of the reference).
// Online softmax in float32 (csrc/kernels/softmax.h:128-186 of the reference); query head h reads KV head
// h / (nh / nkv) (csrc/kernels/flash_fwd_kernel.h:593).  With slopes (one per query head) the score of key j for the
// token at p gains slopes[h] * (j - p), a bias that is linear in the distance (the reference's kernels take such
// slopes too: csrc/kernels/mask.h:155-157, 179-186; its Llama passes none).
// With chunk > 0 the token at p sees only the keys of its own chunk of positions, [(p / chunk) * chunk, p]
// (chunks count from position 0 of the request).  With sinks (one float32 per query head) the softmax denominator
// also holds exp(sinks[h]): a weight that belongs to no key and carries no value.  With keep > 0 a token whose window has
// moved on also sees the first `keep` keys of its request, visited before those of the window.  Values may have another
// number of columns (vd) than keys (hd).
//
// A workgroup takes sixteen rows: the query heads of one KV head (up to sixteen of them) for as many neighbouring tokens
// of the step as that leaves, so that a key or value is fetched once for all of them.  Its waves take blocks of sixteen
// keys (multiples of 16, counted from position 0) in turn and meet in LDS.  Scores and sums are
// v_mfma_f32_16x16x4_f32, true float32: a lane of the score product holds one key's runs of eight columns, as the cache
// lays them out, and MFMA j sums columns 8 g + j over the four lane groups g; its results are four neighbouring keys of
// one row, which is what the lane feeds to the value product, whose other operand is four neighbouring tokens of one
// column: one load of the cache's layout.  Nothing passes LDS but the waves' results.
//
// Measured on MI355X (float32, 32 heads over 8 of 64 columns, four layers; before: a wave per token and head, the values
// read one token and 64 columns at a time, columns 64 bytes apart): 836 tokens of four prompts and sixteen steps of four
// decoded tokens with 40 to 530 keys, 11.8 -> 1.25 ms in all: 63 us a layer for the prompts, 16 for four decoded tokens
// (79 and 28 with loads under conditions, a block's values asked for behind its scores).
// Bound by the chain of page number, keys and values of a wave's few blocks.
#include "common.h"
#include "cache_layout.h"

using namespace atoma;

typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int kMaxHead = 256;
constexpr int kRows = 16;

struct GenericAttnArgs {
  const int32_t* block_tables;
  const int32_t* token_seq;
  const int32_t* positions;
  const float* slopes;
  const float* sinks;
  int q_stride, out_stride, max_blocks, n_tokens, nh, nkv, hd, vd, page_size, window, chunk, keep, tokens;
  float scale;
};

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const f32x4 lo = *reinterpret_cast<const f32x4*>(p), hi = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = lo[i], v[4 + i] = hi[i];
}
__device__ __forceinline__ void load8(const bf16_t* p, float (&v)[8]) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  const uint32_t q[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) v[2 * i] = __uint_as_float(q[i] << 16), v[2 * i + 1] = __uint_as_float(q[i] & 0xffff0000u);
}
__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return f32x4{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
               __uint_as_float(u.y & 0xffff0000u)};
}

// HB: columns of keys and of values that the registers hold (32, 64, 128 or 256); NW: waves that share the keys.  EXACT: keys
// and values have HB columns and a block of sixteen keys lies in one page, in the MFMA's order: then no load stands under a
// condition, all of a block's are on their way together, and the next block's page numbers with them.
template <int HB, int NW, bool EXACT, typename TQ, typename TC>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(1, HB > 128 ? 1 : 8)))
paged_attention_generic_kernel(const TQ* __restrict__ q, const TC* __restrict__ kcache, const TC* __restrict__ vcache,
                               TQ* __restrict__ out, GenericAttnArgs a) {
  constexpr int KG = HB / 32, VT = HB / 16;
  __shared__ f32x4 part[NW / 2][VT][64];
  __shared__ float part_m[NW / 2][64], part_l[NW / 2][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int group = a.nh / a.nkv, pieces = (group + kRows - 1) / kRows;       // (more than 16 heads a KV head: in pieces)
  const int kvh = blockIdx.y / pieces, h_first = (blockIdx.y % pieces) * kRows;
  const int heads = min(kRows, group - h_first);                              // heads a token has among the rows
  const int t0 = blockIdx.x * a.tokens, t_end = min(t0 + a.tokens, a.n_tokens);
  // this lane's row: a token and a head
  const int my_t = t0 + r16 / heads, h = kvh * group + h_first + r16 % heads;
  const bool real = my_t < t_end;
  const int p = a.positions[real ? my_t : t0];
  int first = (a.window > 0 && p - a.window + 1 > 0) ? p - a.window + 1 : 0;
  if (a.chunk > 0 && (p / a.chunk) * a.chunk > first) first = (p / a.chunk) * a.chunk;
  const float slope = a.slopes ? a.slopes[h] : 0.f;
  const int runs = a.hd / 8;
  const size_t k_tile = (size_t)a.page_size * a.hd, v_tile = (size_t)a.page_size * a.vd;
  const bool whole_runs = EXACT || (a.page_size & 15) == 0;

  float qv[KG][8];
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    const int run = kg + 4 * g;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      qv[g][e] = real && run < runs ? to_f32(q[(size_t)my_t * a.q_stride + (size_t)h * a.hd + run * 8 + e]) : 0.f;
  }

  // the tokens of the rows, request by request: what one holds (infinities, NaN) never meets another's rows
  for (int lo = t0; lo < t_end;) {
    const int s = a.token_seq[lo];
    int hi = lo, p_max = 0, first_min = 0x7fffffff;
    for (; hi < t_end && a.token_seq[hi] == s; ++hi) {
      const int pt = a.positions[hi];
      int ft = (a.window > 0 && pt - a.window + 1 > 0) ? pt - a.window + 1 : 0;
      if (a.chunk > 0 && (pt / a.chunk) * a.chunk > ft) ft = (pt / a.chunk) * a.chunk;
      p_max = max(p_max, pt), first_min = min(first_min, ft);
    }
    const bool mine = real && my_t >= lo && my_t < hi;
    const int32_t* table = a.block_tables + (size_t)s * a.max_blocks;
    const int kept = min(a.keep, first_min);                       // kept keys that no window reaches
    const int kept_blocks = (kept + 15) / 16, from = max(first_min / 16, kept_blocks), last = p_max / 16;
    const int visits = kept_blocks + last - from + 1;

    float m = -INFINITY, l = 0.f;
    f32x4 acc[VT];
#pragma unroll
    for (int v = 0; v < VT; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};

    // keys that nobody here may see are never read: their pages may be another request's by now
    auto exists = [&](int j) { return j <= p_max && (j < kept || j >= first_min); };
    auto base_of = [&](int b) { return 16 * (b < kept_blocks ? b : from + b - kept_blocks); };
    auto key_of = [&](int base) { return exists(base + r16) ? base + r16 : p_max; };
    // page numbers: of the lane's key, and of the block's values
    int k_page = 0, v_page_no = 0;
    auto pages_of = [&](int b) {
      const int base = base_of(b < visits ? b : visits - 1);
      k_page = table[key_of(base) / a.page_size];
      if (whole_runs) v_page_no = table[base / a.page_size];
    };
    pages_of(wave);
    for (int b = wave; b < visits; b += NW) {
      const int base = base_of(b), j_key = key_of(base);
      const TC* kt = kcache + ((size_t)k_page * a.nkv + kvh) * k_tile + (size_t)(j_key % a.page_size) * 8;
      const size_t v_page = ((size_t)v_page_no * a.nkv + kvh) * v_tile;
      const int v_off = whole_runs ? base % a.page_size : 0;
      f32x4 vv[VT];
      float kv[KG][8];
      if constexpr (EXACT) {
#pragma unroll
        for (int g = 0; g < KG; ++g) load8(kt + (size_t)(kg + 4 * g) * a.page_size * 8, kv[g]);
#pragma unroll
        for (int v = 0; v < VT; ++v) vv[v] = load4(vcache + v_page + value_offset(v * 16 + r16, v_off + 4 * kg, HB, 16));
      }
      pages_of(b + NW);
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < KG; ++g) {
        if constexpr (!EXACT) {
          const int run = kg + 4 * g;
#pragma unroll
          for (int e = 0; e < 8; ++e) kv[g][e] = 0.f;
          if (run < runs) load8(kt + (size_t)run * a.page_size * 8, kv[g]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[g][e], qv[g][e], sc, 0, 0, 0);
      }
      // the lane's four keys of row r16
      bool vis[4], all_seen = true, all_there = true;
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = base + 4 * kg + i;
        vis[i] = mine && j <= p && (j >= first || j < a.keep);
        all_seen = all_seen && (vis[i] || !mine), all_there = all_there && exists(j);
        sc[i] = vis[i] ? sc[i] * a.scale + slope * (float)(j - p) : -INFINITY;
        mx = fmaxf(mx, sc[i]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m, mx);
      const float corr = m_new == -INFINITY ? 1.f : expf(m - m_new);
      f32x4 pj;
#pragma unroll
      for (int i = 0; i < 4; ++i) pj[i] = vis[i] ? expf(sc[i] - m_new) : 0.f;
      l = l * corr + (pj[0] + pj[1] + pj[2] + pj[3]);
      m = m_new;
      // the lane's column of every sixteen, tokens 4 kg .. + 3
      const bool all_rows = __all(all_seen);
      bool finite = true;
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const int d = v * 16 + r16;
        if constexpr (!EXACT) vv[v] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (EXACT || d < a.vd) {
          if (whole_runs) {
            if constexpr (!EXACT) vv[v] = load4(vcache + v_page + value_offset(d, v_off + 4 * kg, a.vd, a.page_size));
            if (!all_there) {
#pragma unroll
              for (int i = 0; i < 4; ++i) vv[v][i] = exists(base + 4 * kg + i) ? vv[v][i] : 0.f;
            }
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = base + 4 * kg + i;
              if (exists(j))
                vv[v][i] = to_f32(vcache[((size_t)table[j / a.page_size] * a.nkv + kvh) * v_tile +
                                         value_offset(d, j % a.page_size, a.vd, a.page_size)]);
            }
          }
        }
        if (!all_rows) {
#pragma unroll
          for (int i = 0; i < 4; ++i) finite = finite && fabsf(vv[v][i]) < INFINITY;
        }
        acc[v] *= corr;
      }
      if (all_rows || __all(finite)) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int v = 0; v < VT; ++v)
            acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[v][e], pj[e], acc[v], 0, 0, 0);
      } else {
        // a value that is no finite number, behind a mask: its weight of zero would still make it a NaN for rows that
        // do not see it, so the block's keys are added one by one, to the rows that do
        for (int i = 0; i < 16; ++i) {
          const int j = base + i;
          if (!exists(j)) continue;
          const float w = __shfl(i % 4 == 0 ? pj[0] : i % 4 == 1 ? pj[1] : i % 4 == 2 ? pj[2] : pj[3], (i / 4) * 16 + r16, 64);
          const bool sees = mine && j <= p && (j >= first || j < a.keep);
          const TC* vt = vcache + ((size_t)table[j / a.page_size] * a.nkv + kvh) * v_tile;
#pragma unroll
          for (int v = 0; v < VT; ++v)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int d = v * 16 + 4 * kg + e;
              if (sees && d < a.vd) acc[v][e] += w * to_f32(vt[value_offset(d, j % a.page_size, a.vd, a.page_size)]);
            }
        }
      }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);

    // the waves meet, halves at a time
#pragma unroll
    for (int half = NW / 2; half > 0; half >>= 1) {
      __syncthreads();
      if (wave >= half && wave < 2 * half) {
        part_m[wave - half][lane] = m, part_l[wave - half][lane] = l;
#pragma unroll
        for (int v = 0; v < VT; ++v) part[wave - half][v][lane] = acc[v];
      }
      __syncthreads();
      if (wave < half) {
        const float m_o = part_m[wave][lane], m_new = fmaxf(m, m_o);
        const float c = m_new == -INFINITY ? 1.f : expf(m - m_new), c_o = m_new == -INFINITY ? 0.f : expf(m_o - m_new);
        l = l * c + part_l[wave][lane] * c_o;
        m = m_new;
#pragma unroll
        for (int v = 0; v < VT; ++v) acc[v] = acc[v] * c + part[wave][v][lane] * c_o;
      }
    }
    if (wave == 0 && mine) {
      if (a.sinks) {
        // the sink joins the denominator under the common maximum
        const float sk = a.sinks[h], m_new = fmaxf(m, sk), corr = expf(m - m_new);
        l = l * corr + expf(sk - m_new);
#pragma unroll
        for (int v = 0; v < VT; ++v) acc[v] *= corr;
      }
      const float inv = 1.0f / l;  // at least the token's own key is visible, so l > 0
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = v * 16 + 4 * kg + e;
          if (d < a.vd) out[(size_t)my_t * a.out_stride + (size_t)h * a.vd + d] = from_f32<TQ>(acc[v][e] * inv);
        }
    }
    lo = hi;
  }
}

template <int HB, typename TQ, typename TC>
static void launch_generic(const TQ* q, const TC* kcache, const TC* vcache, TQ* out, GenericAttnArgs a, bool one_each,
                           hipStream_t stream) {
  const int group = a.nh / a.nkv, pieces = (group + kRows - 1) / kRows;
  // (decode steps have another request in every token: a token a workgroup, and eight waves for its keys)
  a.tokens = one_each ? 1 : group >= kRows ? 1 : kRows / group;
  const dim3 grid((a.n_tokens + a.tokens - 1) / a.tokens, a.nkv * pieces);
  const bool exact = a.hd == HB && a.vd == HB && a.page_size % 16 == 0;
  const bool many = (size_t)grid.x * grid.y >= 512;
#define ATOMA_GEN(NW, E)                                                                                                  \
  hipLaunchKernelGGL((paged_attention_generic_kernel<HB, NW, E, TQ, TC>), grid, dim3(64 * NW), 0, stream, q, kcache, vcache, \
                     out, a)
  // (wide heads hold more registers than eight waves a workgroup have)
  if constexpr (HB <= 64) {
    if (!many && exact) ATOMA_GEN(8, true);
    else if (!many) ATOMA_GEN(8, false);
    else if (exact) ATOMA_GEN(4, true);
    else ATOMA_GEN(4, false);
  } else {
    (void)many;
    if (exact) ATOMA_GEN(4, true);
    else ATOMA_GEN(4, false);
  }
#undef ATOMA_GEN
}

extern "C" int atoma_paged_attention_generic(const void* q, int q_stride, const void* kcache, const void* vcache,
                                             void* out, int out_stride, int act_dtype, int cache_dtype,
                                             const int32_t* block_tables, int max_blocks, const int32_t* token_seq,
                                             const int32_t* positions, float scale, int window, int page_size,
                                             int n_tokens, int nh, int nkv, int hd, const float* slopes,
                                             int chunk, const float* sinks, int keep, int vd, hipStream_t stream) {
  if (n_tokens <= 0) return 0;
  if (hd <= 0 || hd > kMaxHead || vd <= 0 || vd > kMaxHead || keep < 0 || nkv <= 0 || nh % nkv || page_size <= 0 || max_blocks <= 0 || nh > 65535)
    return ATOMA_ERR_SHAPE;
  GenericAttnArgs a = {block_tables, token_seq, positions, slopes, sinks, q_stride, out_stride, max_blocks, n_tokens, nh,
                       nkv, hd, vd, page_size, window, chunk, keep, 1, scale};
  const int cols = hd > vd ? hd : vd;
  const bool one_each = n_tokens <= 64;      // (few tokens: more workgroups matter more than shared keys)
#define ATOMA_ATTN(TQ, TC)                                                                                             \
  do {                                                                                                                 \
    const TQ* q_ = (const TQ*)q;                                                                                       \
    const TC *k_ = (const TC*)kcache, *v_ = (const TC*)vcache;                                                         \
    if (cols <= 32) launch_generic<32, TQ, TC>(q_, k_, v_, (TQ*)out, a, one_each, stream);                             \
    else if (cols <= 64) launch_generic<64, TQ, TC>(q_, k_, v_, (TQ*)out, a, one_each, stream);                        \
    else if (cols <= 128) launch_generic<128, TQ, TC>(q_, k_, v_, (TQ*)out, a, one_each, stream);                      \
    else launch_generic<256, TQ, TC>(q_, k_, v_, (TQ*)out, a, one_each, stream);                                       \
  } while (0)
  if (act_dtype == kF32 && cache_dtype == kF32) ATOMA_ATTN(float, float);
  else if (act_dtype == kBF16 && cache_dtype == kBF16) ATOMA_ATTN(bf16_t, bf16_t);
  else if (act_dtype == kF32 && cache_dtype == kBF16) ATOMA_ATTN(float, bf16_t);
  else if (act_dtype == kBF16 && cache_dtype == kF32) ATOMA_ATTN(bf16_t, float);
  else return ATOMA_ERR_DTYPE;
#undef ATOMA_ATTN
  ATOMA_LAUNCH_CHECK();
  return 0;
}
