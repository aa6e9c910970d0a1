// bfloat16 x bfloat16 products on the matrix cores for many rows of activations (prompts, large batches):
// X[M, K] * W[N, K]^T with float32 accumulation, in tiles of BM rows of X against BN rows of W a workgroup.
//
// Bound by the matrix cores, and behind them by LDS: a wave's tile of TM x TN blocks of 16 x 16 reads 1 KB of LDS a block
// row and block column for TM * TN MFMAs.  So tiles are as large as the launch allows (256 x 256 by eight waves), and:
//
//   * both operands go from memory to LDS directly (buffer_load ... lds, 16 bytes a lane), S buffers of 64 values of K in
//     turn, so that no register holds them on the way and S - 1 steps are in flight while one is multiplied;
//   * a row of a buffer is 128 bytes and its eight 16-byte pieces lie in the order piece ^ (row % 8): a wave's LDS reads
//     (16 rows, four pieces) then fall on different banks.  The loads do the permuting: lane l of a load fetches piece
//     (l % 8) ^ (l / 8) of its row, since what it stores is always in lane order;
//   * a step's fragments of 32 values of K are read while the MFMAs of the 32 before run, across the end of the step
//     too: one barrier a step stands between the reads of its last fragments and those of the next step's first, with
//     MFMAs on either side of it;
//   * the first operand of the MFMA is W, so a lane's four results are neighbouring columns of one row of X: two pairs
//     of a rotation, or (with W's rows in blocks of 16 gate rows and their 16 up rows) gate and up of the same output;
//   * workgroups are numbered so that each of the eight XCDs, which take them in turn, gets a run of tiles that lie
//     in a patch of four rows of tiles: its L2 then serves most of what they share (the gate-up product of Llama 1B
//     with 2,048 rows 125 -> 119 us against rows of eight, its down product 72 -> 67).
//
// What leaves: float32 (whole, or a plane a K slice), the float32 residual rows with the sums added, silu(gate) * up in
// bfloat16, or q rotated in bfloat16 and k, v in the paged cache.
//
// Needs K % 64 == 0, N % 16 == 0 and 16-byte aligned rows; the host wrapper checks and otherwise refuses.
#include <type_traits>

#include "common.h"
#include "rope_store.h"

using namespace atoma;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) void* lds_ptr;

enum Epilogue : int { kOutF32 = 0, kOutResid = 1, kOutSilu = 2, kOutRope = 3 };

struct TileOut {
  void* c;               // float32 [slices][M][ldc], the float32 residual rows [M][ldc], or bfloat16 [M][ldc]
  int ldc;
  size_t plane;          // elements between the planes of two K slices
  RopeArgs rope;
};

// Rows of X in groups, each against a weight of its own (experts): a row of tiles is one entry of a list (group, first row),
// a group's rows end where the next one's begin, and the float32 result of row `place` goes, times scale, to the row of its
// slot: choice slot % top of token slot / top, in plane slot % top of plane_rows rows.
struct Groups {
  const int32_t* tiles;      // [max_tiles][2]; group -1: nothing
  const int32_t* offsets;    // [groups + 1]
  const int32_t* perm;       // [places]: the place's slot
  const float* scale;        // [slots] or null
  int top, plane_rows;
};

// BM x BN: a workgroup's tile; WM x WN: its waves; S: LDS buffers.
template <int BM_, int BN_, int WM_, int WN_, int S_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_, NW = WM * WN;
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;                  // blocks of 16 of a wave
  static constexpr int QX = BM / 8, XI = (QX + NW - 1) / NW;                  // loads of eight rows: a step's, a wave's
  static constexpr int QW = BN / 8, WI = (QW + NW - 1) / NW;
  static constexpr int XBUF = BM * 128, BUF = (BM + BN) * 128, LDS = S * BUF;  // bytes; X's rows, then W's
  // what a wave may still have on its way when the next step has to be there: the S - 2 steps behind it
  static constexpr int NEWER = (S - 2) * (XI + WI);
  static_assert(S >= 3 && LDS <= 160 * 1024 && NEWER + XI + WI < 64, "");
};

// silu(g) * u, as exact as g / (1 + expf(-g)) * u (measured over |g| <= 88: the same largest and mean error, 1.8e-7 and 3e-8
// of the value).  The division's range is known, so a reciprocal and one correction of the quotient do, at a quarter of numerator
// and denominator, which keeps the reciprocal of any finite denominator a normal number; div_fixup sets infinities and
// NaN right.  2,048 rows against 16,384 x 2,048: 102.5 us, 105.1 with the compiler's division, 97.8 with the hardware's exponential
// of the rounded -g log2 e, whose result was off by up to 1.8e-6 (4e-7 in the mean for g below -5).
__device__ __forceinline__ float silu_times(float g, float u) {
  const float e = expf(-g), den = fmaf(e, 0.25f, 0.25f), num = g * 0.25f;
  const float y = __builtin_amdgcn_rcpf(den), q = num * y;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-den, q, num), y, q), 1.0f + e, g) * u;
}

constexpr int kPatch = 4;      // rows of tiles in a patch

#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t rsrc_t;

template <typename C>
struct Frag { bf16x8 w[C::TN], x[C::TM]; };

// Q loads of eight rows, I of them this wave's (one that has less than others repeats the last: the same bytes to the same
// place)
template <int Q, int I, int NW>
__device__ __forceinline__ void issue(char* __restrict__ dst, rsrc_t src, int k, const uint32_t (&vo)[I], int wave) {
#pragma unroll
  for (int i = 0; i < I; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)(dst + min(i * NW + wave, Q - 1) * 1024), 16, vo[i], k, 0, 0);
}

template <typename C>
__device__ __forceinline__ void read(const char* __restrict__ rd, int half, uint32_t xr, uint32_t wr, int lane, Frag<C>& f) {
  const uint32_t col = (uint32_t)((half * 4 + (lane >> 4)) ^ (lane & 7)) * 16;
#pragma unroll
  for (int i = 0; i < C::TN; ++i) f.w[i] = *reinterpret_cast<const bf16x8*>(rd + wr + i * 2048 + col);
#pragma unroll
  for (int j = 0; j < C::TM; ++j) f.x[j] = *reinterpret_cast<const bf16x8*>(rd + xr + j * 2048 + col);
}

template <typename C>
__device__ __forceinline__ void multiply(const Frag<C>& f, f32x4 (&acc)[C::TN][C::TM]) {
#pragma unroll
  for (int j = 0; j < C::TM; ++j)
#pragma unroll
    for (int i = 0; i < C::TN; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[i], f.x[j], acc[i][j], 0, 0, 0);
}

// a read of LDS behind every few MFMAs
template <typename C>
__device__ __forceinline__ void interleave() {
  constexpr int reads = C::TM + C::TN, per = C::TM * C::TN / reads > 0 ? C::TM * C::TN / reads : 1;
#pragma unroll
  for (int i = 0; i < reads; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, per, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x8, C::TM * C::TN, 0);
}

// Step s behind its barrier: f1 holds the last fragments of step s, rd is the buffer of step s + 1, wr that of step s, which
// nobody reads any more and which the loads of step s + S (at byte k of the rows) go to.  (That the two pointers promise
// not to overlap is what keeps the compiler from waiting for those loads before the reads.)
template <typename C>
__device__ __forceinline__ void step(const char* __restrict__ rd, char* __restrict__ wr, bool more, rsrc_t xb, rsrc_t wb, int k,
                                     const uint32_t (&xo)[C::XI], const uint32_t (&wo)[C::WI], int wave, uint32_t xr, uint32_t wrow,
                                     int lane, Frag<C>& f0, Frag<C>& f1, f32x4 (&acc)[C::TN][C::TM]) {
  read<C>(rd, 0, xr, wrow, lane, f0);
  multiply<C>(f1, acc);
  interleave<C>();
  __builtin_amdgcn_sched_barrier(0);
  // (the loads wait until the first fragments' reads are out: 2,048 rows, N 3,072, K 8,192 by tiles of 256 x 128 111 -> 104 us)
  if (more) {
    issue<C::QX, C::XI, C::NW>(wr, xb, k, xo, wave);
    issue<C::QW, C::WI, C::NW>(wr + C::XBUF, wb, k, wo, wave);
  }
  read<C>(rd, 1, xr, wrow, lane, f1);
  multiply<C>(f0, acc);
  interleave<C>();
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// The rotary epilogue of a wave's tile of ROWS x COLS sums, which lie in LDS row by row: rows from m0, columns from n0.
// (Written out for the sums in registers, with four-byte stores and a trip to memory for every row's position and slot, it
// took 13 us of 43 for Llama 1B with 2,048 rows; 9 of 37 now.)
//   q and k: a lane takes sixteen columns of a row, eight rotation pairs: columns 2 i, 2 i + 1 become columns i of the
//     head's lower and of its upper half; eight and eight of them leave as 16 bytes each, to the query's row or to the runs
//     of the key tile, which holds a token's columns in eights;
//   values: a lane takes a column of four rows; where those are neighbours in the value tile they leave together.
// (hd is a multiple of 16, so sixteen columns from a multiple of 16 on lie in one head.)
// Lane r holds row r's position, page and place in the page (page < 0: no cache write), asked for before the product: a trip
// to memory every time round the loops is what they cannot afford.
template <int ROWS, int COLS>
__device__ __forceinline__ void rope_tile(const float* __restrict__ sums, int m0, int M, int n0, int N, int pos_of, int page_of,
                                          int off_of, const RopeArgs& ra, uint16_t* __restrict__ q_out, int ldq, int lane) {
  static_assert(ROWS <= 64, "a lane a row");
  const int hd = ra.hd, half = hd >> 1, rotated = (ra.nh + ra.nkv) * hd;
  constexpr int BLOCKS = COLS / 16;
  const int live = min(BLOCKS, (N - n0) / 16), turned = min(live, max(0, rotated - n0) / 16);       // (N >= n0 here)
#pragma unroll 1
  for (int first = 0; first < ROWS * turned; first += 64) {
    const int item = first + lane, r = item / turned, b = item - r * turned, m = m0 + r;
    const int pos = __shfl(pos_of, r, 64), page = __shfl(page_of, r, 64), off = __shfl(off_of, r, 64);
    if (r >= ROWS || m >= M) continue;
    const int n = n0 + b * 16, head = n / hd, i0 = (n - head * hd) >> 1;
    const f32x4* const cp = reinterpret_cast<const f32x4*>(ra.cos_t + (size_t)pos * half + i0);
    const f32x4* const sp = reinterpret_cast<const f32x4*>(ra.sin_t + (size_t)pos * half + i0);
    const f32x4 c[2] = {cp[0], cp[1]}, sn[2] = {sp[0], sp[1]};
    const f32x4* const x = reinterpret_cast<const f32x4*>(sums + r * COLS + b * 16);
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const f32x4 v = x[p];
      const float c0 = c[p >> 1][(p & 1) * 2], c1 = c[p >> 1][(p & 1) * 2 + 1], s0 = sn[p >> 1][(p & 1) * 2], s1 = sn[p >> 1][(p & 1) * 2 + 1];
      lo[p] = pack_bf16(v[0] * c0 - v[1] * s0, v[2] * c1 - v[3] * s1);
      hi[p] = pack_bf16(v[1] * c0 + v[0] * s0, v[3] * c1 + v[2] * s1);
    }
    if (head >= ra.nh && page < 0) continue;
    uint16_t *to, *to_hi;
    if (head < ra.nh) {
      to = q_out + (size_t)m * ldq + (size_t)head * hd + i0;
      to_hi = to + half;
    } else {
      uint16_t* const tile = ra.kcache + ((size_t)page * ra.nkv + (head - ra.nh)) * ra.page_size * hd;
      to = tile + key_offset(off, i0, ra.page_size);
      to_hi = tile + key_offset(off, i0 + half, ra.page_size);
    }
    *reinterpret_cast<uint4*>(to) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    *reinterpret_cast<uint4*>(to_hi) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  }
  if (turned >= live) return;
  const int columns = (live - turned) * 16;
#pragma unroll 1
  for (int first = 0; first < ROWS / 4 * columns; first += 64) {
    const int item = first + lane, r = item / columns * 4, cc = item - item / columns * columns;
    int page[4], off[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) page[t] = __shfl(page_of, r + t, 64), off[t] = __shfl(off_of, r + t, 64);
    if (r >= ROWS || m0 + r >= M) continue;
    const int n = n0 + turned * 16 + cc, head = (n - rotated) / hd, d = n - rotated - head * hd;
    uint16_t v[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = (uint16_t)pack_bf16(sums[(r + t) * COLS + turned * 16 + cc], 0.f);
    auto place = [&](int t) {
      return ra.vcache + ((size_t)page[t] * ra.nkv + head) * ra.page_size * hd + value_offset(d, off[t], hd, ra.page_size);
    };
    if ((ra.page_size & 3) == 0 && page[0] >= 0 && (off[0] & 3) == 0 && page[1] == page[0] && page[2] == page[0] &&
        page[3] == page[0] && off[1] == off[0] + 1 && off[2] == off[0] + 2 && off[3] == off[0] + 3) {
      *reinterpret_cast<uint2*>(place(0)) = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (page[t] >= 0) *place(t) = v[t];
    }
  }
}

// at most n loads of this wave still on their way; reads: and none of its LDS reads
template <int N, bool READS>
__device__ __forceinline__ void wait() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((READS ? 0 : 15) << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
#endif

#if defined(__HIP_DEVICE_COMPILE__)
// What leaves of row m: NB blocks of 16 columns from column nw on, of which this lane has columns 4 kg .. + 3.
template <int EPI, bool GROUPED, int NB>
__device__ __forceinline__ void put_row(const f32x4 (&v)[NB], int m, int nw, int N, int kg, const TileOut& out, const Groups& groups) {
  size_t to_row = 0;
  float to_scale = 1.f;
  if constexpr (EPI == kOutF32 && GROUPED) {
    const int slot = groups.perm[m];
    to_row = (size_t)(slot % groups.top) * groups.plane_rows + slot / groups.top;
    if (groups.scale) to_scale = groups.scale[slot];
  }
  if constexpr (EPI == kOutSilu) {
    uint16_t* const row = (uint16_t*)out.c + (size_t)m * out.ldc;
#pragma unroll
    for (int i = 0; i + 1 < NB; i += 2) {         // blocks of 16 gate rows, then the 16 up rows of the same outputs
      if (nw + i * 16 >= N) continue;
      const int n = (nw + i * 16) / 2 + kg * 4;
      uint2 r;
      __bf16* const o = reinterpret_cast<__bf16*>(&r);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (__bf16)silu_times(v[i][e], v[i + 1][e]);
      *reinterpret_cast<uint2*>(row + n) = r;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int n = nw + i * 16 + kg * 4;
      if (nw + i * 16 >= N) continue;                // (N is a multiple of 16: a block is there or is not)
      if constexpr (EPI == kOutF32 && GROUPED) {
        *reinterpret_cast<f32x4*>((float*)out.c + to_row * out.ldc + n) = v[i] * to_scale;
      } else if constexpr (EPI == kOutF32) {
        *reinterpret_cast<f32x4*>((float*)out.c + blockIdx.y * out.plane + (size_t)m * out.ldc + n) = v[i];
      } else {
        f32x4* const p = reinterpret_cast<f32x4*>((float*)out.c + (size_t)m * out.ldc + n);
        *p = *p + v[i];
      }
    }
  }
}

// The workgroup's tile: this XCD's run of the order, patches of kPatch rows of tiles, column by column.
template <typename C>
__device__ __forceinline__ void tile_of(int rows, int N, int& mi, int& n0) {
  const int mt = (rows + C::BM - 1) / C::BM, nt = (N + C::BN - 1) / C::BN;
  const int share = (mt * nt) >> 3, rest = (mt * nt) & 7, xcd = blockIdx.x & 7;
  const int id = xcd * share + min(xcd, rest) + (blockIdx.x >> 3);
  const int patch = id / (kPatch * nt), pm = min(kPatch, mt - patch * kPatch), in = id - patch * kPatch * nt;
  mi = patch * kPatch + in % pm, n0 = (in / pm) * C::BN;
}
#endif

// (rows: M of X, or the entries of the groups' list times BM)
template <typename C, int EPI, bool GROUPED>
__global__ void __launch_bounds__(64 * C::NW, C::NW >= 8 ? 2 : 1)
gemm_tile_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int rows, int N, int ldx, int ldw, int k_len,
                 TileOut out, Groups groups) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  int mi, n0;
  tile_of<C>(rows, N, mi, n0);
  const int k0 = blockIdx.y * k_len;
  int m0 = mi * C::BM, M = rows;
  if constexpr (GROUPED) {
    const int g = groups.tiles[2 * mi];
    if (g < 0) return;
    m0 = groups.tiles[2 * mi + 1], M = groups.offsets[g + 1];
    w += (size_t)g * N * ldw;
  }

  const int rows_x = min(C::BM, M - m0), rows_w = min(C::BN, N - n0);
  // (rows past the end: the last one, never stored)
  const int lr = lane >> 3;
  const uint32_t piece = ((lane & 7) ^ lr) * 16;
  uint32_t xo[C::XI], wo[C::WI];
#pragma unroll
  for (int i = 0; i < C::XI; ++i) xo[i] = (uint32_t)min(min(i * C::NW + wave, C::QX - 1) * 8 + lr, rows_x - 1) * ldx * 2 + piece;
#pragma unroll
  for (int i = 0; i < C::WI; ++i) wo[i] = (uint32_t)min(min(i * C::NW + wave, C::QW - 1) * 8 + lr, rows_w - 1) * ldw * 2 + piece;
  const rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)m0 * ldx + k0), 0, ((rows_x - 1) * ldx + k_len) * 2, 0x00027000);
  const rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * ldw + k0), 0, ((rows_w - 1) * ldw + k_len) * 2, 0x00027000);

  f32x4 acc[C::TN][C::TM];
#pragma unroll
  for (int i = 0; i < C::TN; ++i)
#pragma unroll
    for (int j = 0; j < C::TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = wave / C::WN, wn = wave % C::WN;
  const uint32_t xr = (wm * (C::BM / C::WM) + r16) * 128, wr = C::XBUF + (wn * (C::BN / C::WN) + r16) * 128;

  int pos_of = 0, page_of = -1, off_of = 0;
  if constexpr (EPI == kOutRope) {
    const int row = m0 + wm * (C::BM / C::WM) + lane;
    if (lane < C::BM / C::WM && row < M) {
      const int slot = out.rope.slot_mapping[row];
      pos_of = out.rope.positions[row];
      if (slot >= 0) page_of = slot / out.rope.page_size, off_of = slot - page_of * out.rope.page_size;
    }
  }

  const int steps = k_len / 64;
#pragma unroll
  for (int s = 0; s < C::S; ++s)
    if (s < steps) {
      issue<C::QX, C::XI, C::NW>(lds + s * C::BUF, xb, s * 128, xo, wave);
      issue<C::QW, C::WI, C::NW>(lds + s * C::BUF + C::XBUF, wb, s * 128, wo, wave);
    }
  if (C::S <= steps) wait<C::NEWER + C::XI + C::WI, false>();
  else wait<0, false>();
  meet();
  Frag<C> f0, f1;
  read<C>(lds, 0, xr, wr, lane, f0);
  read<C>(lds, 1, xr, wr, lane, f1);
  multiply<C>(f0, acc);
  int cur = 0, nxt = C::BUF;
  for (int s = 0; s + 1 < steps; ++s) {
    // step s + 1 has landed, for this wave here and for all behind the barrier, and so are all reads of step s done
    if (s + C::S <= steps) wait<C::NEWER, true>();
    else wait<0, true>();
    meet();
    step<C>(lds + nxt, lds + cur, s + C::S < steps, xb, wb, (s + C::S) * 128, xo, wo, wave, xr, wr, lane, f0, f1, acc);
    cur = nxt;
    nxt = nxt + C::BUF == C::LDS ? 0 : nxt + C::BUF;
  }
  multiply<C>(f1, acc);

  if constexpr (EPI == kOutRope) {
    constexpr int ROWS = C::TM * 16, COLS = C::TN * 16;
    static_assert(ROWS * COLS * 4 * C::NW <= 160 * 1024, "");
    wait<0, true>();
    meet();                  // everybody's reads of the last step are done
    float* const sums = reinterpret_cast<float*>(lds) + wave * (ROWS * COLS);
#pragma unroll
    for (int j = 0; j < C::TM; ++j)
#pragma unroll
      for (int i = 0; i < C::TN; ++i) *reinterpret_cast<f32x4*>(sums + (j * 16 + r16) * COLS + i * 16 + kg * 4) = acc[i][j];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int nw = n0 + wn * COLS;
    if (nw < N) rope_tile<ROWS, COLS>(sums, m0 + wm * ROWS, M, nw, N, pos_of, page_of, off_of, out.rope,
                                          (uint16_t*)out.c, out.ldc, lane);
    return;
  }
#pragma unroll
  for (int j = 0; j < C::TM; ++j) {
    const int m = m0 + wm * (C::BM / C::WM) + j * 16 + r16;
    if (m >= M) continue;
    f32x4 v[C::TN];
#pragma unroll
    for (int i = 0; i < C::TN; ++i) v[i] = acc[i][j];
    put_row<EPI, GROUPED>(v, m, n0 + wn * (C::BN / C::WN), N, kg, out, groups);
  }
#endif
}

// ---- tiles in phases ------------------------------------------------------------------------------------------------------
// With one barrier a step a buffer is free, and the loads for the step after next can start, only when all of its fragments have been
// read, and those loads must be there a step later: 64 KB of a burst and the latency behind it for a tile of 256 x 256, 1.27 us a step on
// their own, about what a step's MFMAs take.  Here a step is multiplied in four phases, half of X's rows by half of W's at a time, and a
// phase's fragments are read under the MFMAs of the one before:
//   X0 W0 (W1 is read), X0 W1 (X1), X1 W1 (the next step's X0, into the registers of this one's), X1 W0 (its W0, into W1's)
// So X0 and W0 of a step are read before the step begins, W1 and X1 by its middle, and with a barrier at either place the halves are
// loaded anew a step and a half before they are read again, 32 KB at a time: the loads alone take 0.95 us a step.
// us, before / now, on their own: gate-up with SiLU, 2,048 rows against 16,384 x 2,048 116 / 111, 16,384 x 3,072 164 / 156, 28,672 x 4,096
// 391 / 370; in a program's steps 106 to 123, 149 and 355.  float32 sums of 8,192^3 800 / 763.  What is left is power: the MFMAs alone would
// take 555 of the 763 and the loads alone 486, with all of them served by the L2 the product still takes 735, and the clock is at 1.85 GHz;
// priorities for the MFMAs (s_setprio) cost 2 %.
//
// Two buffers instead of three or four also leave half of a CU's LDS to a second workgroup where a tile has 128 rows: one workgroup's first
// loads and its results then pass under the other's products, and a barrier holds up half of a CU's waves.  Against tiles of the same 256 or
// 128 rows with one barrier a step, four buffers and a workgroup a CU (some 18,000 products; geometric means of the time, by workgroups
// a CU up to one / more): 128 x 128 0.95 to 0.98 (see kLongSteps) / 0.84 to 0.89, 256 x 128 0.97 / 0.98, 128 x 192 against 256 x 96 0.92 to 0.97 / 0.85 to
// 0.88, 128 x 64 1.01 / 0.83 to 0.88 (so only there).  us, before / now: q, k, v of 2,048 rows against 3,072 x 2,048 35.9 / 33.0 (one round
// of 128 x 192, which keeps one barrier a step: 31.1), two slices of 2,048 x 8,192 69.0 / 65.3.  (192 x 128, patches of eight rows of tiles and 128 x 160 gave nothing; 256 x 160 by halves of 80 lost 1 %.)
// EU: waves a SIMD that the registers are to leave room for (four: two workgroups of eight waves).
template <int BM_, int BN_, int WM_, int WN_, int EU_ = 2>
struct Phased {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NW = WM * WN, EU = EU_;
  static constexpr int XH = BM / 2, WH = BN / 2;                              // rows of a half
  static constexpr int JX = XH / WM / 16, JW = WH / WN / 16;                  // blocks of 16 of a wave in a half
  static constexpr int QX = XH / 8, XI = (QX + NW - 1) / NW;                  // loads of eight rows: a half's, a wave's
  static constexpr int QW = WH / 8, WI = (QW + NW - 1) / NW;
  static constexpr int PAIR = XI + WI;                                        // of a wave for a half of X and one of W
  static constexpr int X0 = 0, X1 = XH * 128, W0 = BM * 128, W1 = W0 + WH * 128;      // bytes: the halves of a buffer
  static constexpr int BUF = (BM + BN) * 128, LDS = 2 * BUF;
  static_assert(XH % (16 * WM) == 0 && WH % (16 * WN) == 0 && LDS <= 160 * 1024 && 4 * PAIR < 64, "");
};

#if defined(__HIP_DEVICE_COMPILE__)
template <int NB>
__device__ __forceinline__ void read_half(const char* __restrict__ p, uint32_t row, int lane, bf16x8 (&f)[NB][2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t col = (uint32_t)((h * 4 + (lane >> 4)) ^ (lane & 7)) * 16;
#pragma unroll
    for (int i = 0; i < NB; ++i) f[i][h] = *reinterpret_cast<const bf16x8*>(p + row + i * 2048 + col);
  }
}
// READS reads of LDS spread over the MFMAs
template <int READS, int JW, int JX>
__device__ __forceinline__ void phase(const bf16x8 (&w)[JW][2], const bf16x8 (&x)[JX][2], f32x4 (&acc)[JW][JX]) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < JX; ++j)
#pragma unroll
      for (int i = 0; i < JW; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][h], x[j][h], acc[i][j], 0, 0, 0);
  constexpr int all = 2 * JW * JX, per = all / READS > 0 ? all / READS : 1;
#pragma unroll
  for (int i = 0; i < READS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x8, per, 0);
  }
  __builtin_amdgcn_sched_group_barrier(0x8, all, 0);
  __builtin_amdgcn_sched_barrier(0);
}
#endif

// Two steps or more; ODD: their number is (a kernel that takes either spills registers; of these only 128 x 192 with the rotary end, whose four waves
// a SIMD leave 128, does: one a lane, outside the loop).
template <typename C, int EPI, bool GROUPED, bool ODD>
__global__ void __launch_bounds__(64 * C::NW, C::EU)
gemm_phased_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int rows, int N, int ldx, int ldw, int k_len,
                   TileOut out, Groups groups) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  int mi, n0;
  tile_of<C>(rows, N, mi, n0);
  const int k0 = blockIdx.y * k_len;
  int m0 = mi * C::BM, M = rows;
  if constexpr (GROUPED) {
    const int g = groups.tiles[2 * mi];
    if (g < 0) return;
    m0 = groups.tiles[2 * mi + 1], M = groups.offsets[g + 1];
    w += (size_t)g * N * ldw;
  }
  const int rows_x = min(C::BM, M - m0), rows_w = min(C::BN, N - n0);
  // a half's rows through a buffer of its own: what lies past the last row is out of its range, reads as zero and is never stored.  A second
  // half without a row is the first one's first row: no load has a place in K beyond the end of its buffer.  (All of its rows again, which are on
  // their way from the same lines already, made tiles of 256 x 128 with 65 to 128 rows 1.05 (sums) and 1.11 (SiLU) times as long as by one
  // barrier a step, over 59 products; now 0.97 and 0.99.)
  const int lr = lane >> 3;
  const uint32_t piece = ((lane & 7) ^ lr) * 16;
  uint32_t xo[C::XI], wo[C::WI];
#pragma unroll
  for (int i = 0; i < C::XI; ++i) xo[i] = (uint32_t)(min(i * C::NW + wave, C::QX - 1) * 8 + lr) * ldx * 2 + piece;
#pragma unroll
  for (int i = 0; i < C::WI; ++i) wo[i] = (uint32_t)(min(i * C::NW + wave, C::QW - 1) * 8 + lr) * ldw * 2 + piece;
  auto half = [&](const uint16_t* p, int ld, int there) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, ((there - 1) * ld + k_len) * 2, 0x00027000);
  };
  const uint16_t* const xp = x + (size_t)m0 * ldx + k0;
  const uint16_t* const wp = w + (size_t)n0 * ldw + k0;
  const int x1 = rows_x > C::XH ? C::XH : 0, w1 = rows_w > C::WH ? C::WH : 0;
  const rsrc_t xb0 = half(xp, ldx, min(rows_x, C::XH)), xb1 = half(xp + (size_t)x1 * ldx, ldx, max(1, rows_x - C::XH));
  const rsrc_t wb0 = half(wp, ldw, min(rows_w, C::WH)), wb1 = half(wp + (size_t)w1 * ldw, ldw, max(1, rows_w - C::WH));

  f32x4 acc[2][2][C::JW][C::JX];          // by half of W, half of X
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < C::JW; ++i)
#pragma unroll
        for (int j = 0; j < C::JX; ++j) acc[g][h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wm = wave / C::WN, wn = wave % C::WN;
  const uint32_t xr = (wm * (C::XH / C::WM) + r16) * 128, wr = (wn * (C::WH / C::WN) + r16) * 128;

  // lanes from 0 on: the wave's rows of X's first half, then those of the second
  constexpr int ROWS = C::XH / C::WM;
  int pos_of = 0, page_of = -1, off_of = 0;
  if constexpr (EPI == kOutRope) {
    static_assert(2 * ROWS <= 64 && (ROWS & (ROWS - 1)) == 0, "a lane a row");
    const int row = m0 + lane / ROWS * C::XH + wm * ROWS + lane % ROWS;
    if (lane < 2 * ROWS && row < M) {
      const int slot = out.rope.slot_mapping[row];
      pos_of = out.rope.positions[row];
      if (slot >= 0) page_of = slot / out.rope.page_size, off_of = slot - page_of * out.rope.page_size;
    }
  }

  const int steps = k_len / 64;
  auto load_first = [&](char* __restrict__ buf, int s) {
    issue<C::QX, C::XI, C::NW>(buf + C::X0, xb0, s * 128, xo, wave);
    issue<C::QW, C::WI, C::NW>(buf + C::W0, wb0, s * 128, wo, wave);
  };
  auto load_second = [&](char* __restrict__ buf, int s) {
    issue<C::QW, C::WI, C::NW>(buf + C::W1, wb1, s * 128, wo, wave);
    issue<C::QX, C::XI, C::NW>(buf + C::X1, xb1, s * 128, xo, wave);
  };
  char* const b0 = lds;
  char* const b1 = lds + C::BUF;
  load_first(b0, 0);
  load_second(b0, 0);
  load_first(b1, 1);
  load_second(b1, 1);
  wait<3 * C::PAIR, false>();
  meet();
  bf16x8 fx0[C::JX][2], fx1[C::JX][2], fa[C::JW][2], fb[C::JW][2];
  read_half(b0 + C::X0, xr, lane, fx0);
  read_half(b0 + C::W0, wr, lane, fa);
  // Step s, whose X0 and W0 are in fx0 and w0.  REST: how many steps are behind it (2: two or more).  (now and own are the same buffer,
  // then the other one: that they promise not to overlap keeps the compiler from waiting for the loads before the reads.)
  auto step = [&](auto rest, int s, const char* __restrict__ now, char* __restrict__ own, const char* __restrict__ then,
                  bf16x8 (&w0)[C::JW][2], bf16x8 (&w1)[C::JW][2]) {
    constexpr int REST = decltype(rest)::value;
    // everybody has read X0 and W0, and this step's W1 and X1 have landed
    if constexpr (REST > 0) wait<2 * C::PAIR, true>();
    else wait<0, true>();
    meet();
    read_half(now + C::W1, wr, lane, w1);
    if constexpr (REST == 2) load_first(own, s + 2);
    phase<2 * C::JW>(w0, fx0, acc[0][0]);
    read_half(now + C::X1, xr, lane, fx1);
    phase<2 * C::JX>(w1, fx0, acc[1][0]);
    // everybody has read W1 and X1, and the next step's X0 and W0 have landed
    if constexpr (REST > 0) {
      wait<(REST == 2 ? 2 : 1) * C::PAIR, true>();
      meet();
      read_half(then + C::X0, xr, lane, fx0);
    }
    if constexpr (REST == 2) load_second(own, s + 2);
    phase<2 * C::JX>(w1, fx1, acc[1][1]);
    if constexpr (REST > 0) read_half(then + C::W0, wr, lane, w1);
    phase<2 * C::JW>(w0, fx1, acc[0][1]);
  };
  constexpr std::integral_constant<int, 0> none{};
  constexpr std::integral_constant<int, 1> one{};
  constexpr std::integral_constant<int, 2> more{};
  int s = 0;
  for (; s + 2 + ODD < steps; s += 2) {
    step(more, s, b0, b0, b1, fa, fb);
    step(more, s + 1, b1, b1, b0, fb, fa);
  }
  if constexpr (ODD) {
    step(more, s, b0, b0, b1, fa, fb);
    step(one, s + 1, b1, b1, b0, fb, fa);
    step(none, s + 2, b0, b0, b1, fa, fb);
  } else {
    step(one, s, b0, b0, b1, fa, fb);
    step(none, s + 1, b1, b1, b0, fb, fa);
  }
  if constexpr (EPI == kOutRope) {
    // (all sums at once do not fit LDS: a half of X's rows by a half of W's at a time.  2,048 rows against 6,144 x 4,096: 256 tiles of 256 x
    // 192, 86 us on their own, 95 in the steps of a long prompt; by 256 x 96 103, by the library with the rotation's kernel behind it 93)
    constexpr int COLS = C::WH / C::WN;
    wait<0, true>();
    meet();                  // everybody's reads of the last step are done
    float* const sums = reinterpret_cast<float*>(lds) + wave * (ROWS * COLS);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int from = h * ROWS + lane % ROWS, pos = __shfl(pos_of, from, 64), page = __shfl(page_of, from, 64), off = __shfl(off_of, from, 64);
#pragma unroll
      for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int j = 0; j < C::JX; ++j)
#pragma unroll
          for (int i = 0; i < C::JW; ++i)
            *reinterpret_cast<f32x4*>(sums + (j * 16 + r16) * COLS + i * 16 + kg * 4) = acc[g][h][i][j];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        const int nw = n0 + g * C::WH + wn * COLS;
        if (nw < N) rope_tile<ROWS, COLS>(sums, m0 + h * C::XH + wm * ROWS, M, nw, N, pos, page, off, out.rope, (uint16_t*)out.c, out.ldc, lane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
      }
    }
    return;
  }
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < C::JX; ++j) {
      const int m = m0 + h * C::XH + wm * (C::XH / C::WM) + j * 16 + r16;
      if (m >= M) continue;
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        f32x4 v[C::JW];
#pragma unroll
        for (int i = 0; i < C::JW; ++i) v[i] = acc[g][h][i][j];
        put_row<EPI, GROUPED>(v, m, n0 + g * C::WH + wn * (C::WH / C::WN), N, kg, out, groups);
      }
    }
#endif
}

template <typename C, int EPI, bool GROUPED, bool ODD>
static int launch_phased(const void* x, const void* w, int M, int N, int K, int ldx, int ldw, int slices, const TileOut& out,
                         hipStream_t stream, const Groups& groups) {
  // (every device that the kernel is launched on has its own setting)
  const hipError_t e = hipFuncSetAttribute((const void*)gemm_phased_kernel<C, EPI, GROUPED, ODD>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  if (e != hipSuccess) return (int)e;
  const int64_t tiles = (int64_t)((M + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN);
  if (tiles > 0x7fffffff) return ATOMA_ERR_SHAPE;
  hipLaunchKernelGGL((gemm_phased_kernel<C, EPI, GROUPED, ODD>), dim3((int)tiles, slices), dim3(64 * C::NW), C::LDS, stream,
                     (const uint16_t*)x, (const uint16_t*)w, M, N, ldx, ldw, K / slices, out, groups);
  ATOMA_LAUNCH_CHECK();
  return 0;
}
template <typename C, int EPI, bool GROUPED = false>
static int launch(const void* x, const void* w, int M, int N, int K, int ldx, int ldw, int slices, const TileOut& out,
                  hipStream_t stream, const Groups& groups = Groups{}) {
  // (every device that the kernel is launched on has its own setting)
  constexpr int lds = EPI == kOutRope && C::BM * C::BN * 4 > C::LDS ? C::BM * C::BN * 4 : C::LDS;      // (the rotary epilogue's sums)
  const hipError_t e = hipFuncSetAttribute((const void*)gemm_tile_kernel<C, EPI, GROUPED>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  if (e != hipSuccess) return (int)e;
  const int64_t tiles = (int64_t)((M + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN);
  if (tiles > 0x7fffffff) return ATOMA_ERR_SHAPE;
  hipLaunchKernelGGL((gemm_tile_kernel<C, EPI, GROUPED>), dim3((int)tiles, slices), dim3(64 * C::NW), lds, stream,
                     (const uint16_t*)x, (const uint16_t*)w, M, N, ldx, ldw, K / slices, out, groups);
  ATOMA_LAUNCH_CHECK();
  return 0;
}

// (one step: by a tile of as many rows with one barrier a step)
template <typename C, int EPI, bool GROUPED = false>
static int launch_phased(const void* x, const void* w, int M, int N, int K, int ldx, int ldw, int slices, const TileOut& out,
                         hipStream_t stream, const Groups& groups = Groups{}) {
  const int steps = K / slices / 64;
  if (steps == 1) return launch<Tile<C::BM, 128, C::BM / 64, 2, 3>, EPI, GROUPED>(x, w, M, N, K, ldx, ldw, slices, out, stream, groups);
  return steps % 2 ? launch_phased<C, EPI, GROUPED, true>(x, w, M, N, K, ldx, ldw, slices, out, stream, groups)
                   : launch_phased<C, EPI, GROUPED, false>(x, w, M, N, K, ldx, ldw, slices, out, stream, groups);
}

constexpr int kCUs = 256;

// Tiles of which a CU can hold two where they go in phases, which is the quicker way once there is more than one for a CU.  One for each CU has
// its LDS for four buffers: 128 x 64 takes 1.00 to 1.04 times as long in phases then, 128 x 192 with a long end 1.00 to 1.02, and 128 x 128 with
// residual rows, 0.98 on its own, 1.02 within a prompt's steps; with other ends 0.95 to 0.98, but beyond kLongSteps steps of K, where the loads set
// the pace all the way, 1.00 to 1.02 and from 97 on 1.03 (sums, rotary) and 1.04 (SiLU), up to 1.15 (137 products).
constexpr int kLongSteps = 64;
// (kernels/gemm_bf16.py: _rounds counts with the same line)
static bool two_a_cu(int M, int N, int bm, int bn, int slices) {
  return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * slices > kCUs;
}

template <int EPI>
static int pick(int tile, const void* x, const void* w, int M, int N, int K, int ldx, int ldw, int slices, const TileOut& out,
                hipStream_t stream) {
  constexpr bool GATED = EPI == kOutSilu, STORES = EPI == kOutResid || EPI == kOutRope;
  (void)GATED;
#define ATOMA_TILE(...) return launch<Tile<__VA_ARGS__>, EPI>(x, w, M, N, K, ldx, ldw, slices, out, stream)
#define ATOMA_PHASED(...) return launch_phased<Phased<__VA_ARGS__>, EPI>(x, w, M, N, K, ldx, ldw, slices, out, stream)
  switch (tile) {
    case 0: if constexpr (EPI != kOutRope) ATOMA_PHASED(256, 256, 2, 4); break;                  // (its sums do not fit LDS)
    case 1: ATOMA_PHASED(256, 128, 4, 2);
    // by four waves, whose larger shares read less LDS, or eight where the end is long, which gain by 2 to 13 percent there
    case 2:
      if ((EPI == kOutResid || K / slices / 64 > kLongSteps) && !two_a_cu(M, N, 128, 128, slices)) ATOMA_TILE(128, 128, 2, 4, 4);
      if constexpr (STORES) ATOMA_PHASED(128, 128, 2, 4, 4);
      else ATOMA_PHASED(128, 128, 2, 2);
    case 3:
      if (two_a_cu(M, N, 128, 64, slices)) ATOMA_PHASED(128, 64, 4, 1, 4);
      ATOMA_TILE(128, 64, 2, 2, 4);
    case 4: if constexpr (!GATED) ATOMA_TILE(256, 160, 4, 2, 3); break;     // (a wave's blocks are not in pairs)
    case 5:
      if constexpr (STORES) {
        if (two_a_cu(M, N, 128, 192, slices)) ATOMA_PHASED(128, 192, 4, 2, 4);
        ATOMA_TILE(128, 192, 2, 4, 4);
      } else if constexpr (!GATED) {
        ATOMA_PHASED(128, 192, 2, 2);
      }
      break;
    // 33 to 64 rows, and q, k, v and small weights with some hundred: bound by what a CU brings to LDS, so small tiles, two workgroups a CU, and K in slices.  64 rows, gate-up
    // of 16,384 x 2,048 in 64 x 64 17.7 us with four buffers, 18.8 with three, 18.2 with eight (one workgroup a CU); 64 x 128 with three
    // 21.6.  Planes of 3,072 x 8,192 13.7 by 64 x 128 in eight slices, 15.4 by 64 x 64.
    case 6: if constexpr (EPI == kOutF32 || GATED) ATOMA_TILE(64, 64, 2, 2, 4); break;
    case 7: if constexpr (EPI == kOutF32) ATOMA_TILE(64, 128, 2, 2, 3); break;
    case 8: if constexpr (EPI == kOutRope) ATOMA_PHASED(256, 192, 4, 2); break;
  }
#undef ATOMA_TILE
#undef ATOMA_PHASED
  return ATOMA_ERR_SHAPE;
}

// x [M, K] and w [N, K] bfloat16.  kind: what leaves (see Epilogue); tile: which of the tiles above; slices: parts of K, a
// float32 plane each (kind 0 only).  rope: positions, cos_t, sin_t, kcache, vcache, slot_mapping and sizes (kind 3 only).
extern "C" int atoma_gemm_tile(const void* x, const void* w, void* c, int kind, int tile, int M, int N, int K, int ldx,
                               int ldw, int ldc, int slices, const int32_t* positions, const float* cos_t, const float* sin_t,
                               void* kcache, void* vcache, const int32_t* slot_mapping, int page_size, int nh, int nkv, int hd, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || slices <= 0 || K % (64 * slices) || N % 16 || ldx < K || ldw < K || ldx % 8 || ldw % 8 || ldx > (1 << 21) ||
      ldw > (1 << 21) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) || (slices > 1 && kind != kOutF32) || slices > 65535 || ldc % 4 ||
      ((uintptr_t)c & (kind == kOutF32 || kind == kOutResid ? 15 : 7)))
    return ATOMA_ERR_SHAPE;
  TileOut out{c, ldc, (size_t)M * ldc, 
              RopeArgs{positions, cos_t, sin_t, (uint16_t*)kcache, (uint16_t*)vcache, slot_mapping, page_size, nh, nkv, hd}};
  if (kind == kOutRope) {
    if (N != (nh + 2 * nkv) * hd || hd % 16 || ldc < nh * hd || nh <= 0 || nkv <= 0 || page_size <= 0 || !positions || !cos_t ||
        !sin_t || !kcache || !vcache || !slot_mapping || ldc % 8 ||
        (((uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)c | (uintptr_t)cos_t | (uintptr_t)sin_t) & 15))
      return ATOMA_ERR_SHAPE;
    return pick<kOutRope>(tile, x, w, M, N, K, ldx, ldw, 1, out, stream);
  }
  if (kind == kOutSilu) {
    if (N % 32 || ldc < N / 2) return ATOMA_ERR_SHAPE;
    return pick<kOutSilu>(tile, x, w, M, N, K, ldx, ldw, 1, out, stream);
  }
  if (ldc < N) return ATOMA_ERR_SHAPE;
  if (kind == kOutF32) return pick<kOutF32>(tile, x, w, M, N, K, ldx, ldw, slices, out, stream);
  if (kind == kOutResid) return pick<kOutResid>(tile, x, w, M, N, K, ldx, ldw, 1, out, stream);
  return ATOMA_ERR_SHAPE;
}

// The same for rows in groups (see Groups): x [places, K], w [groups, N, K], tiles [max_tiles][2] for tiles of the rows that
// `tile` has.  kind 0: float32 planes by slot, [top][plane_rows][N]; kind 2: silu(gate) * up, bfloat16 [places, N / 2].
extern "C" int atoma_gemm_tile_groups(const void* x, const void* w, void* c, int kind, int tile, int N, int K, const int32_t* tiles,
                                      int max_tiles, const int32_t* offsets, const int32_t* perm, const float* scale, int top,
                                      int plane_rows, hipStream_t stream) {
  if (max_tiles <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 64 || N % 32 || K > (1 << 21) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)c & 15) ||
      max_tiles > (1 << 20) || top <= 0 || plane_rows <= 0 || (kind == kOutSilu && scale != nullptr))
    return ATOMA_ERR_SHAPE;
  const TileOut out{c, kind == kOutSilu ? N / 2 : N, 0, RopeArgs{}};
  const Groups groups{tiles, offsets, perm, scale, top, plane_rows};
#define ATOMA_GROUPS(HOW, BM, ...)                                                                                        \
  do {                                                                                                                     \
    if (kind == kOutSilu)                                                                                                  \
      return HOW<__VA_ARGS__, kOutSilu, true>(x, w, max_tiles * BM, N, K, K, K, 1, out, stream, groups);                  \
    if (kind == kOutF32)                                                                                                   \
      return HOW<__VA_ARGS__, kOutF32, true>(x, w, max_tiles * BM, N, K, K, K, 1, out, stream, groups);                   \
  } while (0)
  switch (tile) {
    case 0: ATOMA_GROUPS(launch_phased, 256, Phased<256, 256, 2, 4>); break;
    case 1: ATOMA_GROUPS(launch_phased, 256, Phased<256, 128, 4, 2>); break;
    case 2: ATOMA_GROUPS(launch_phased, 128, Phased<128, 128, 2, 2>); break;
    case 3:
      if (two_a_cu(max_tiles * 128, N, 128, 64, 1)) ATOMA_GROUPS(launch_phased, 128, Phased<128, 64, 4, 1, 4>);
      else ATOMA_GROUPS(launch, 128, Tile<128, 64, 2, 2, 4>);
      break;
  }
#undef ATOMA_GROUPS
  return ATOMA_ERR_SHAPE;
}
