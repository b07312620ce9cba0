// The PLE block's projections (engraft/replica/layers.py:594-606: key = emb
// w_key^T and value = emb w_value^T, as two column groups over the same A in
// one launch, and their backward d_emb = d_key w_key + d_value w_value as two
// K segments with the weights' transposes kept row-major):
//
//   C[M, N] (+)= A[M, K] B[N, K]^T  (+ A2[M, K2] B2[N, K2]^T)
//
// in two arithmetics.
//
// gemm_x3_kernel, fp32 on the bf16 matrix cores: each fp32 operand is split
// once (eg_split_bf16) into bf16 planes hi = rne(x) and lo = rne(x - hi)
// (x - hi is exact in fp32), and C accumulates hi*hi + hi*lo + lo*hi in fp32
// on v_mfma_f32_32x32x16_bf16.  hi + lo keeps 16 of fp32's 24 mantissa bits,
// so each product carries a relative error up to ~3 x 2^-18 (fp32's own is
// 2^-24): about 1e-5 of the result on random data, at the bf16 rate.
//
// gemm_f32_kernel, fp32 arithmetic on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32): the products of an fp32 matmul, each operand
// read once as fp32.
//
// Tiling, both: 256 x 256 output tiles, one workgroup a CU; K in steps of 32
// through a two-stage LDS ring filled by direct-to-LDS loads
// (global_load_lds_dwordx4: lane i of a wavefront writes 16 bytes at the
// wavefront's LDS base + 16 i), so the next step's loads are in flight during
// the current step's MFMAs without passing through registers.
// gemm_x3: eight wavefronts of 128 x 64 outputs (4 x 2 MFMA tiles of 32 x 32),
// 128 KB of LDS (four bf16 planes a stage), software-pipelined: a half step's
// fragments are read during the other half step's MFMAs, one barrier a step.
// On the key projection (M 2048, N 10240, K 2560) 290 us against 319 us for
// the 128 x 128 tiles of four wavefronts it replaces (two workgroups a CU,
// the last round in K quarters), and the backward's d_emb 400 against 470 us;
// sixteen wavefronts of 64 x 64 or eight of 64 x 128 ran 1-4 % slower, four
// of 128 x 128 (one a SIMD, the accumulators in the accumulation registers,
// a third less LDS read a step) 8-13 % slower on the bf16x3 and bf16x6 shapes, the
// same tile without the pipelining 2 % slower, with 2-way LDS bank conflicts
// on the fragment reads 2-3 % slower; the reads interleaved one by one with
// the MFMAs, or the wave priority raised over the MFMA passes, within 1 %.  Measured earlier on the 128 x 128 tile
// and dropped: three stages, scheduling hints, register-staged loads into a
// padded LDS tile (20 % slower).  Counters on the key projection: the matrix
// cores busy 55 % of the cycles (SQ_VALU_MFMA_BUSY_CYCLES) at a shader clock
// of ~1.8 GHz under this load.  gemm_f32: sixteen wavefronts of 64 x 64, 128 KB of
// LDS: 88.8 % of the fp32 MFMA peak where the tiles fill whole rounds,
// against 83.3 % for 128 x 128 tiles of four.
//
// The last round.  When the tile count leaves the last round (one tile a CU)
// partly empty, the (tile, K step) units of that round's tiles are cut into
// one contiguous range a CU, each range's parts (one or two tiles) go to a
// workspace, and sk_sum_kernel adds each tile's parts in K order into C, so
// the result does not depend on scheduling.  On MI355X (256 CUs): the fp32
// key + value's 400 tiles run as 256 whole and 144 in 256 ranges of 45 of a
// tile's 80 K steps (1040 us against 1249 us whole and 1126 us with the 144
// in sevenths), the backward's 80 tiles of 400 K steps in 256 ranges of 125
// (1018 us against 1091 us in thirds); the bf16x3 key projection's 320 tiles
// as 256 whole and 64 in 256 ranges of 20.  An explicit k_slices cuts every
// tile into that many equal pieces instead (piece_sum_kernel adds them).
//
// Workgroups are dispatched round-robin over the 8 XCDs; the whole tiles are
// remapped so that each XCD takes a contiguous run of tiles, grouped 8 row
// tiles deep, whose A and B panels its own L2 shares.
#include "eg_common.h"

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

namespace eg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroupM = 8;
constexpr int kXcds = 8;
constexpr int kBK = 32;
constexpr int kStages = 2;

// gemm_x3's tile: 256 x 256 outputs of 2 x 4 wavefronts of 128 x 64; two
// stages of four 256 x 32 bf16 planes, 128 KB of LDS
constexpr int kX3BM = 256, kX3BN = 256, kX3WM = 2, kX3WN = 4;

// What both kernels share: output, tiles and the whole-tile / piece split.
struct Plan {
  int64_t kt0;            // K steps of segment 0
  int64_t kt_total;
  int64_t kt_per_piece;
  int dp_tiles;           // blocks [0, dp_tiles) run whole tiles (logical tiles 0 .. dp_tiles-1)
  int pieces;             // pieces per remaining tile; block dp_tiles + q runs piece q
  int sk_groups;          // > 0: the remaining tiles' K steps in sk_groups contiguous ranges instead
  int64_t sk_units;       //      (tiles - dp_tiles) x kt_total (tile, K step) units split among them
  float* c[2];            // per column group
  int64_t ldc[2];
  float* ws;              // [tiles - dp_tiles][pieces][tile] partial products, or [2 sk_groups][tile]
  int64_t m, n[2];
  int tiles_m, tiles_n0, tiles_n;
  int accumulate;         // 1: C += result
};

struct GemmSeg {
  const __bf16* a_hi;
  const __bf16* a_lo;
  const __bf16* b_hi[2];  // per column group
  const __bf16* b_lo[2];
  int64_t lda, ldb[2];    // in bf16, multiples of 8
  int64_t ktiles;         // K / 32
};

struct GemmArgs {
  GemmSeg seg[2];
  int n_seg;
  Plan p;
};

struct F32Seg {
  const float* a;
  const float* b[2];      // per column group
  int64_t lda, ldb[2];    // in floats, multiples of 4
  int64_t ktiles;         // K / 32
};

struct F32Args {
  F32Seg seg[2];
  int n_seg;
  Plan p;
};

// hi = rne(x), lo = rne(x - hi) for 4 values.
__device__ inline void split4(const float4 v, bf16x4& hi, bf16x4& lo) {
  hi[0] = (__bf16)v.x;
  hi[1] = (__bf16)v.y;
  hi[2] = (__bf16)v.z;
  hi[3] = (__bf16)v.w;
  lo[0] = (__bf16)(v.x - (float)hi[0]);
  lo[1] = (__bf16)(v.y - (float)hi[1]);
  lo[2] = (__bf16)(v.z - (float)hi[2]);
  lo[3] = (__bf16)(v.w - (float)hi[3]);
}

// x [rows, cols] (row stride ld) -> hi, lo [rows, kp] with kp = cols rounded up
// to 32 and the padding zero; blockIdx.y walks rows, each thread 4 values.
// With a third plane lo2 (bf16x6's split): hi, mid = lo as above, and
// lo2 = rne(x - hi - lo) (both differences exact in fp32).
template <bool VEC, bool THREE>
__global__ __launch_bounds__(256) void split_kernel(const float* __restrict__ x, int64_t rows, int64_t cols,
                                                    int64_t ld, int64_t kp, __bf16* __restrict__ hi,
                                                    __bf16* __restrict__ lo, __bf16* __restrict__ lo2) {
  const int64_t c = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= kp) return;
  for (int64_t r = blockIdx.y; r < rows; r += gridDim.y) {
    const float* src = x + r * ld + c;
    float4 v;
    if (VEC && c + 3 < cols) {
      v = *(const float4*)src;
    } else {
      v.x = c + 0 < cols ? src[0] : 0.0f;
      v.y = c + 1 < cols ? src[1] : 0.0f;
      v.z = c + 2 < cols ? src[2] : 0.0f;
      v.w = c + 3 < cols ? src[3] : 0.0f;
    }
    bf16x4 h, l;
    split4(v, h, l);
    *(bf16x4*)(hi + r * kp + c) = h;
    *(bf16x4*)(lo + r * kp + c) = l;
    if constexpr (THREE) {
      bf16x4 l2;
      l2[0] = (__bf16)((v.x - (float)h[0]) - (float)l[0]);
      l2[1] = (__bf16)((v.y - (float)h[1]) - (float)l[1]);
      l2[2] = (__bf16)((v.z - (float)h[2]) - (float)l[2]);
      l2[3] = (__bf16)((v.w - (float)h[3]) - (float)l[3]);
      *(bf16x4*)(lo2 + r * kp + c) = l2;
    }
  }
}

// Logical tile -> (row tile, column tile): groups of kGroupM row tiles, each
// group walked column tile by column tile.
__device__ inline void grouped(int logical, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int in_group = kGroupM * tiles_n;
  const int g = logical / in_group;
  const int first_m = g * kGroupM;
  const int gsize = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
  const int r = logical % in_group;
  tm = first_m + r % gsize;
  tn = r / gsize;
}

// The block's work: a whole tile (piece < 0) or piece `piece` of a tile of the
// last round, its K steps [kv0, kv1), and where its output goes.
struct Work {
  int64_t m0, n0, kv0, kv1;
  int grp, piece;
};

// Block b of nb whole-tile blocks -> logical tile: block b runs on XCD b % 8,
// and each XCD takes a contiguous run of tiles.
__device__ inline int xcd_order(int b, int nb) {
  const int x = b % kXcds, i = b / kXcds;
  const int per = nb / kXcds, extra = nb % kXcds;
  return x * per + (x < extra ? x : extra) + i;
}

// The work of one tile (logical index) over K steps [kv0, kv1).
template <int BM, int BN>
__device__ inline Work tile_work(const Plan& p, int logical, int64_t kv0, int64_t kv1, int piece) {
  Work w;
  int tm, tn;
  grouped(logical, p.tiles_m, p.tiles_n, tm, tn);
  w.grp = tn < p.tiles_n0 ? 0 : 1;
  w.m0 = (int64_t)tm * BM;
  w.n0 = (int64_t)(w.grp ? tn - p.tiles_n0 : tn) * BN;
  w.kv0 = kv0;
  w.kv1 = kv1;
  w.piece = piece;
  return w;
}

// An output's value from its sum: the sum itself ...
struct NoScale {
  __device__ float operator()(float v, int, int64_t, int64_t) const { return v; }
};
// ... or the sum times the powers of two its operands' rows were divided by.
struct RowScale {
  const int32_t* a;      // exponent of A's row
  const int32_t* b[2];   // of B's row, per column group
  __device__ float operator()(float v, int grp, int64_t row, int64_t col) const {
    return ldexpf(v, a[row] + b[grp][col]);
  }
};

// Range s of the last round's (tile, K step) units: [U s / G, U (s + 1) / G).
__device__ inline int64_t sk_start(const Plan& p, int64_t s) { return p.sk_units * s / p.sk_groups; }

// D of a 32 x 32 MFMA tile: lane l holds column l % 32 and rows
// 8 (r / 4) + 4 (l / 32) + r % 4; wavefront (wm, wn) holds TI x TJ such
// tiles, the block of 32 TI x 32 TJ outputs at (32 TI wm, 32 TJ wn) of the
// tile.  A whole tile goes to C (bounded by m and n, added to when
// accumulating); a piece to its BM x BN workspace slot.  `scale` gives an
// output its value from the sum (NoScale: the sum itself); pieces keep sums.
template <int BM, int BN, int TI, int TJ, typename Scale>
__device__ inline void store_acc(const Plan& p, const Work& w, const f32x16 (&acc)[TI][TJ], int wm, int wn,
                                 int lane, const Scale& scale) {
  // the store addresses depend on the lane only; an opaque copy of it keeps the
  // compiler from computing them once ahead of a loop over tiles and holding
  // them (in scratch) across the K loops
  asm volatile("" : "+v"(lane));
  const int r0 = wm * 32 * TI, c0 = wn * 32 * TJ;
  if (w.piece >= 0) {
    float* t = p.ws + (int64_t)w.piece * (BM * BN);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int lc = c0 + j * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          t[(r0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * BN + lc] = acc[i][j][r];
      }
    return;
  }
  float* out = p.c[w.grp];
  const int64_t ld = p.ldc[w.grp], n_grp = p.n[w.grp];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      const int64_t col = w.n0 + c0 + j * 32 + (lane & 31);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = w.m0 + r0 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row < p.m && col < n_grp) {
          float* q = out + row * ld + col;
          const float v = scale(acc[i][j][r], w.grp, row, col);
          *q = p.accumulate ? *q + v : v;
        }
      }
    }
}

__device__ inline int swz(int row, int chunk) { return chunk ^ ((row >> 2) & 3); }
__device__ inline int swz8(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// s_waitcnt vmcnt(0), leaving the other counters alone.
__device__ inline void wait_vm0() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); }
// s_waitcnt vmcnt(N) (N < 16) and s_waitcnt lgkmcnt(0), each alone.
template <int N>
__device__ inline void wait_vm() {
  static_assert(N >= 0 && N < 16, "vmcnt field");
  __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8) | N);
}
__device__ inline void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xf | (7 << 4) | (3 << 14)); }

// Both GEMM kernels walk their blocks the same way: every block covers a range
// [u0, u1) of (tile, K step) units from tile `base` on.  A whole tile is
// [0, kt) of its own tile; piece q of the equal cuts is its K steps of tile
// dp_tiles + q / pieces; with ranges (sk_groups > 0), range s of the last
// round covers units [start(s), start(s + 1)) of the tiles from dp_tiles on.
// A range is shorter than a tile's K steps (the last round has fewer tiles
// than there are ranges), so it meets one or two tiles, t0 and t1 = t0 + 1
// from base, and the block runs the two parts one after the other.  A part of
// a tile goes to workspace slot `slot0` + (its tile - t0).  (Written out in
// each kernel: as a shared helper the fp32 kernel ran 10 % slower.)
#define EG_GEMM_WALK(...)                                                                               \
  const Plan& p = args.p;                                                                               \
  const int64_t kt = p.kt_total;                                                                        \
  const int b = (int)blockIdx.x;                                                                        \
  int base, slot0 = 0;                                                                                  \
  int64_t u0 = 0, u1 = kt;                                                                              \
  if (b < p.dp_tiles) {                                                                                 \
    base = xcd_order(b, p.dp_tiles);                                                                    \
  } else if (p.sk_groups == 0) {                                                                        \
    const int q = b - p.dp_tiles;                                                                       \
    base = p.dp_tiles + q / p.pieces;                                                                   \
    u0 = (int64_t)(q % p.pieces) * p.kt_per_piece;                                                      \
    u1 = u0 + p.kt_per_piece < kt ? u0 + p.kt_per_piece : kt;                                           \
    slot0 = q;                                                                                          \
  } else {                                                                                              \
    const int s = b - p.dp_tiles;                                                                       \
    base = p.dp_tiles;                                                                                  \
    u0 = sk_start(p, s);                                                                                \
    u1 = sk_start(p, s + 1);                                                                            \
    slot0 = 2 * s;                                                                                      \
  }                                                                                                     \
  if (u0 >= u1 && !(u0 == 0 && kt == 0)) return; /* an empty range (no K steps still stores zeros) */  \
  const int64_t t0 = kt > 0 ? u0 / kt : 0, t1 = kt > 0 ? (u1 - 1) / kt : 0;                            \
  _Pragma("unroll 1") for (int64_t t = t0; t <= t1; ++t) {                                              \
    const int64_t k0 = (u0 > t * kt ? u0 : t * kt) - t * kt;                                            \
    const int64_t k1 = (u1 < (t + 1) * kt ? u1 : (t + 1) * kt) - t * kt;                                \
    /* whole: a tile of the full rounds, or one that a range covers from end to end */                  \
    const bool whole = (b < p.dp_tiles || p.sk_groups > 0) && k0 == 0 && k1 == kt;                      \
    const Work w = tile_work<BM, BN>(p, base + (int)t, k0, k1, whole ? -1 : slot0 + (int)(t - t0));     \
    __VA_ARGS__;                                                                                        \
  }

// The products a bf16 GEMM launch adds, over the hi and lo planes it loads
// (a pass: A's lo or hi plane times B's lo or hi plane), the small ones first:
//   PR 3 (bf16x3): lo*hi, hi*lo, hi*hi;
//   PR 4: lo*lo, lo*hi, hi*lo, hi*hi (bf16x6 on the hi and mid planes);
//   PR 2: lo*hi, hi*lo (bf16x6 on the hi and lo planes), passes 1 and 2 of PR 4,
//   which is how gemm_x6_kernel runs them (pass set 4 with a run-time mask).
template <int PR>
__device__ constexpr bool pass_alo(int pass) {
  return PR == 4 ? pass < 2 : pass == 0;
}
template <int PR>
__device__ constexpr bool pass_blo(int pass) {
  return PR == 4 ? (pass == 0 || pass == 2) : pass == 1;
}

// gemm_x3: one tile's (or piece's) K steps [w.kv0, w.kv1) and its store.
// BM x BN tile of WMW x WNW wavefronts, each 32 TI x 32 TJ outputs (TI x TJ
// MFMA tiles).  A stage holds the four bf16 planes ah, al (BM rows) and bh, bl
// (BN rows) of 32 k each, 64 B rows, one after the other; the 16-byte chunk c
// of plane row r sits in slot c ^ ((r >> 2) & 3): a fragment read (16 lanes
// at one chunk of 16 consecutive rows per LDS cycle) then touches 16
// distinct 16-byte bank groups (the counter SQ_LDS_BANK_CONFLICT read half of
// SQ_LDS_IDX_ACTIVE with c ^ ((r >> 1) & 3); 2-3 % faster without the
// conflicts).  A direct-to-LDS load fills 16
// rows of a plane (1 KB), so load q of a stage lands at 16 q rows from the
// stage's start.
// A segment's pass set: PR passes of pass_alo / pass_blo; with RT, only the
// passes whose bit is set in a uniform run-time mask run.
template <int PR, bool RT>
struct PassSet {
  static constexpr int value = PR;
  static constexpr bool masked = RT;
};

template <int BM, int BN, int WMW, int WNW, int PR0, int PR1>
__device__ inline void x3_tile(const GemmArgs& args, const Work& w, __bf16* lds) {
  constexpr int NW = WMW * WNW, TI = BM / WMW / 32, TJ = BN / WNW / 32;
  constexpr int LA = BM / 16, LB = BN / 16;         // loads per A / B plane
  constexpr int LPW = 2 * (LA + LB) / NW;           // loads per wavefront per stage
  constexpr int STAGE = 2 * (BM + BN) * kBK;        // bf16
  static_assert(LA % NW == 0 && LB % NW == 0, "a wavefront's j-th load stays in one plane");
  const Plan& p = args.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = (wave / WNW) * (BM / WMW), c0 = (wave % WNW) * (BN / WNW);
  const int grp = w.grp;
  const int64_t n_grp = p.n[grp];

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // this wavefront's loads per stage: load q = wave + NW j covers plane
  // plane_of(j) (0 ah, 1 al, 2 bh, 3 bl), rows 16 (q - the plane's first load)
  // .. +15; lane i fills row 16 (..) + i / 4, slot i % 4.  Rows past m or n read
  // row m-1 or n-1: their products only reach outputs that are not stored.
  auto plane_of = [](int j) { return NW * j < LA ? 0 : NW * j < 2 * LA ? 1 : NW * j < 2 * LA + LB ? 2 : 3; };
  auto first_of = [](int pl) { return pl == 0 ? 0 : pl == 1 ? LA : pl == 2 ? 2 * LA : 2 * LA + LB; };
  const int uwave = __builtin_amdgcn_readfirstlane(wave);

  // the block's K steps of segment s, whose products are pass set PR
  auto seg_steps = [&](const int s, auto pass_set, const uint32_t live) {
    constexpr int PR = decltype(pass_set)::value, NP = PR;  // passes (products) a half step
    auto on = [&](int pass) { return !decltype(pass_set)::masked || ((live >> pass) & 1u); };
    const int64_t seg0 = s ? p.kt0 : 0, seg1 = s ? p.kt_total : p.kt0;
    const int64_t lo = w.kv0 > seg0 ? w.kv0 : seg0, hi = w.kv1 < seg1 ? w.kv1 : seg1;
    if (lo >= hi) return;
    const GemmSeg& sg = args.seg[s];
    // a load's address: the plane's base (uniform) + a 32-bit byte offset
    // (the host keeps every plane under 4 GiB), one VGPR a load
    // (from an opaque copy of the lane: computed here for the segment, not once
    // for the tile and held across the K loops, which spilled)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    uint32_t off[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      const int pl = plane_of(j), q = uwave + NW * j, row = 16 * (q - first_of(pl)) + (ln >> 2);
      const bool is_a = pl < 2;
      const int64_t gr = (is_a ? w.m0 : w.n0) + row, lim = is_a ? p.m : n_grp;
      const int64_t rr = gr < lim ? gr : lim - 1;
      off[j] = (uint32_t)((rr * (pl < 2 ? sg.lda : sg.ldb[grp]) + swz(row, ln & 3) * 8) * 2);
    }
    auto issue = [&](int64_t kt) {  // K step kt of the segment
      __bf16* st = lds + (kt & 1) * STAGE;
#pragma unroll
      for (int j = 0; j < LPW; ++j) {
        const int pl = plane_of(j), q = uwave + NW * j;
        const __bf16* base = pl == 0 ? sg.a_hi : pl == 1 ? sg.a_lo : pl == 2 ? sg.b_hi[grp] : sg.b_lo[grp];
        __builtin_amdgcn_global_load_lds((const void*)((const char*)(base + kt * kBK) + off[j]),
                                         (__attribute__((address_space(3))) void*)(st + 16 * q * kBK), 16, 0, 0);
      }
    };
    // load j alone: the half step after the barrier issues them one at a time
    // between its MFMAs
    auto issue_one = [&](int64_t kt, int j) {
      __bf16* st = lds + (kt & 1) * STAGE;
      const int pl = plane_of(j), q = uwave + NW * j;
      const __bf16* base = pl == 0 ? sg.a_hi : pl == 1 ? sg.a_lo : pl == 2 ? sg.b_hi[grp] : sg.b_lo[grp];
      __builtin_amdgcn_global_load_lds((const void*)((const char*)(base + kt * kBK) + off[j]),
                                       (__attribute__((address_space(3))) void*)(st + 16 * q * kBK), 16, 0, 0);
    };
    // fragments of half step ks (16 k) of stage kt into set f
    bf16x8 ah[2][TI], al[2][TI], bh[2][TJ], bl[2][TJ];
    auto read = [&](int f, int64_t kt, int ks) {
      const __bf16* st = lds + (kt & 1) * STAGE;
      const int c = ks * 2 + (lane >> 5);
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int ar = r0 + i * 32 + (lane & 31);
        const int ao = ar * kBK + swz(ar, c) * 8;
        ah[f][i] = *(const bf16x8*)(st + ao);
        al[f][i] = *(const bf16x8*)(st + BM * kBK + ao);
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const int br = c0 + j * 32 + (lane & 31);
        const int bo = br * kBK + swz(br, c) * 8;
        bh[f][j] = *(const bf16x8*)(st + 2 * BM * kBK + bo);
        bl[f][j] = *(const bf16x8*)(st + (2 * BM + BN) * kBK + bo);
      }
    };
    // the products of set f, the small ones first, a pass over the TI x TJ
    // tiles each (pass_alo / pass_blo: which planes a pass multiplies)
    auto mfma = [&](int f, int pass) {
      if (!on(pass)) return;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pass_alo<PR>(pass) ? al[f][i] : ah[f][i],
                                                               pass_blo<PR>(pass) ? bl[f][j] : bh[f][j], acc[i][j],
                                                               0, 0, 0);
    };
    // Software pipeline, one barrier a step.  The fragments of one half step
    // are read during the other half step's MFMAs, after its first pass: the
    // compiler's wait for a half step's fragments (it waits for every LDS read
    // issued before it) then comes before the first pass, when only that half
    // step's reads, long issued, are outstanding; and the next reads reuse the
    // registers of the lo*hi pass's lo planes.  The loads of step kt + 2 are
    // issued once every wavefront has read step kt (the barrier in the middle
    // of step kt), a step ahead of their use, spread over the half step after
    // that barrier.
    issue(lo - seg0);
    if (lo + 1 < hi) {
      issue(lo + 1 - seg0);
      wait_vm<LPW>();  // this wavefront's part of the first step is in LDS
    } else {
      wait_vm<0>();
    }
    __builtin_amdgcn_s_barrier();
    read(0, lo - seg0, 0);
    // every step but the last (no branch around the reads)
    for (int64_t kv = lo; kv + 1 < hi; ++kv) {
      const int64_t kt = kv - seg0;
      mfma(0, 0);
      __builtin_amdgcn_sched_barrier(0);  // the reads stay between the passes
      read(1, kt, 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int pass = 1; pass < NP; ++pass) mfma(0, pass);
      __builtin_amdgcn_sched_barrier(0);
      // this wavefront's part of step kt + 1 is in LDS and its reads of step kt
      // are in registers; after the barrier, every wavefront's are
      wait_vm<0>();
      wait_lgkm0();
      __builtin_amdgcn_s_barrier();
      {
        // the second half step's MFMAs (its three passes) with the next half
        // step's fragment reads after the first pass and the loads of step
        // kt + 2 one after every second MFMA: a wavefront's direct-to-LDS loads
        // go out one at a time, and in a burst they held the younger wavefront
        // of each SIMD for ~2,700 cycles without an MFMA (the burst form took
        // 2 % longer a step)
        const bool ld = kv + 2 < hi;
#pragma unroll
        for (int t = 0; t < NP * TI * TJ; ++t) {
          const int pass = t / (TI * TJ), i = (t % (TI * TJ)) / TJ, j = t % TJ;
          if (on(pass))
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pass_alo<PR>(pass) ? al[1][i] : ah[1][i],
                                                               pass_blo<PR>(pass) ? bl[1][j] : bh[1][j], acc[i][j],
                                                               0, 0, 0);
          if (t == TI * TJ - 1) {
            __builtin_amdgcn_sched_barrier(0);
            read(0, kt + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
          if ((t + 1) % 2 == 0 && (t + 1) / 2 - 1 < LPW) {
            __builtin_amdgcn_sched_barrier(0);
            if (ld) issue_one(kt + 2, (t + 1) / 2 - 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
    mfma(0, 0);
    read(1, hi - 1 - seg0, 1);
#pragma unroll
    for (int pass = 1; pass < NP; ++pass) mfma(0, pass);
#pragma unroll
    for (int pass = 0; pass < NP; ++pass) mfma(1, pass);
    __builtin_amdgcn_s_barrier();  // the ring is refilled by the next segment or tile
  };
  // segment by segment (the ring drains at a segment change)
  for (int s = 0; s < args.n_seg; ++s) {
    if constexpr (PR0 == PR1)
      seg_steps(s, PassSet<PR0, false>{}, 0u);
    else  // PR0 4, PR1 2: segment 1 runs passes 1 and 2 of the four (lo*hi, hi*lo)
      seg_steps(s, PassSet<4, true>{}, s ? 0x6u : 0xfu);
  }
  store_acc<BM, BN, TI, TJ>(p, w, acc, wave / WNW, wave % WNW, lane, NoScale{});
}

template <int BM, int BN, int WMW, int WNW, int PR>
__global__ __launch_bounds__(WMW * WNW * 64) void gemm_x3_kernel(const GemmArgs args) {
  extern __shared__ __attribute__((aligned(16))) __bf16 lds[];
  EG_GEMM_WALK(x3_tile<BM, BN, WMW, WNW, PR, PR>(args, w, lds))
}

// bf16x6 of one K segment in one launch: segment 0 is its hi and mid planes
// (the four products of pass set 4), segment 1 the same K over its hi and lo
// planes (lo*hi and hi*lo), both into the same accumulators.
template <int BM, int BN, int WMW, int WNW>
__global__ __launch_bounds__(WMW * WNW * 64) void gemm_x6_kernel(const GemmArgs args) {
  extern __shared__ __attribute__((aligned(16))) __bf16 lds[];
  EG_GEMM_WALK((x3_tile<BM, BN, WMW, WNW, 4, 2>(args, w, lds)))
}

// One MFMA takes one A and one B value per lane (lane l: row / column l % 32,
// k = l / 32), so each lane half works through its own 16 k of a step: lane
// half h reads k 16 h .. 16 h + 15 of its row as four 16-byte chunks and the
// 16 MFMAs of the step pair k = kk (half 0) with k = 16 + kk (half 1).  The
// 16-byte chunk c of tile row r sits in slot c ^ ((r >> 1) & 7): a fragment
// read (16 lanes at one chunk of 16 consecutive rows per LDS cycle) then
// touches 16 distinct 16-byte bank groups.  64 MFMAs of 64 cycles a step
// against 16 KB of LDS reads per wavefront: the matrix cores, not the LDS,
// bound it.  BM x BN tile, (BM / 64) x (BN / 64) wavefronts of 64 x 64; A and
// B tiles of BM and BN rows x 128 B a stage.
// One tile's (or piece's) K steps [w.kv0, w.kv1) and its store.
template <int BM, int BN>
__device__ inline void f32_tile(const F32Args& args, const Work& w, float* ldsf) {
  constexpr int WN = BN / 64, NW = (BM / 64) * WN;
  constexpr int STAGE = (BM + BN) * kBK;           // floats
  constexpr int LPW = (BM + BN) / 8 / NW;          // 8-row loads per wavefront per stage
  constexpr int LA = BM / 8 / NW;                  // of which on A
  static_assert((BM / 8) % NW == 0 && (BN / 8) % NW == 0, "loads per wavefront");
  const Plan& p = args.p;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  const int grp = w.grp;
  const int64_t n_grp = p.n[grp];

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // this wavefront's loads per stage: load q = wave + NW j covers rows 8 q' ..
  // 8 q' + 7 of A (j < LA, q' = q) or B (q' = q - BM / 8); lane i fills row
  // 8 q' + i / 8, slot i % 8.  Rows past m or n read row m-1 or n-1 (not stored).
  const int uwave = __builtin_amdgcn_readfirstlane(wave);

  for (int s = 0; s < args.n_seg; ++s) {
    const int64_t seg0 = s ? p.kt0 : 0, seg1 = s ? p.kt_total : p.kt0;
    const int64_t lo = w.kv0 > seg0 ? w.kv0 : seg0, hi = w.kv1 < seg1 ? w.kv1 : seg1;
    if (lo >= hi) continue;
    const F32Seg& sg = args.seg[s];
    // the load addresses, from an opaque copy of the lane: computed here for the
    // segment rather than once for the tile and held across the K loops (the
    // held form spilled 160 B a lane outside the loop and ran 2-4 % slower)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const float* src[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      const int q = uwave + NW * j, row = 8 * (j < LA ? q : q - BM / 8) + (ln >> 3);
      const int64_t gr = (j < LA ? w.m0 : w.n0) + row, lim = j < LA ? p.m : n_grp;
      src[j] = (j < LA ? sg.a : sg.b[grp]) + (gr < lim ? gr : lim - 1) * (j < LA ? sg.lda : sg.ldb[grp]) +
               swz8(row, ln & 7) * 4;
    }
    auto issue = [&](int64_t kt) {
      float* st = ldsf + (kt & 1) * STAGE;
#pragma unroll
      for (int j = 0; j < LPW; ++j) {
        const int q = uwave + NW * j;
        __builtin_amdgcn_global_load_lds((const void*)(src[j] + kt * kBK),
                                         (__attribute__((address_space(3))) void*)(st + 8 * q * kBK), 16, 0, 0);
      }
    };
    issue(lo - seg0);
    for (int64_t kv = lo; kv < hi; ++kv) {
      const int64_t kt = kv - seg0;
      wait_vm0();
      __builtin_amdgcn_s_barrier();
      const float* st = ldsf + (kt & 1) * STAGE;
      // two halves of the step's 16 k a lane half owns: 8 k (two chunks) of
      // each fragment in registers at a time.  The next step's loads go out
      // after the first half's fragment reads: the wait for them that the
      // compiler puts before the next LDS read (it cannot tell the stages
      // apart) then falls after the first half's MFMAs, not before them.
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float4 fa[2][2], fb[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int ar = wm * 64 + i * 32 + (lane & 31);
          const int br = wn * 64 + i * 32 + (lane & 31);
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const int chunk = 4 * (lane >> 5) + 2 * half + c;
            fa[i][c] = *(const float4*)(st + ar * kBK + swz8(ar, chunk) * 4);
            fb[i][c] = *(const float4*)(st + BM * kBK + br * kBK + swz8(br, chunk) * 4);
          }
        }
        if (half == 0 && kv + 1 < hi) issue(kt + 1);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const float4& av = fa[i][kk >> 2];
              const float4& bv = fb[j][kk >> 2];
              const float x = (kk & 3) == 0 ? av.x : (kk & 3) == 1 ? av.y : (kk & 3) == 2 ? av.z : av.w;
              const float y = (kk & 3) == 0 ? bv.x : (kk & 3) == 1 ? bv.y : (kk & 3) == 2 ? bv.z : bv.w;
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc[i][j], 0, 0, 0);
            }
      }
    }
    __builtin_amdgcn_s_barrier();  // the ring is refilled by the next segment or tile
  }
  store_acc<BM, BN, 2, 2>(p, w, acc, wm, wn, lane, NoScale{});
}

// gemm_f32 over the walk.  The stores' lane addresses are recomputed for
// each part of a range (see store_acc): held across both K loops they spilled
// 62 VGPRs to scratch and cost 4 % on whole tiles.
template <int BM, int BN>
__global__ __launch_bounds__(BM * BN / 64) void gemm_f32_kernel(const F32Args args) {
  extern __shared__ __attribute__((aligned(16))) float ldsf[];
  EG_GEMM_WALK(f32_tile<BM, BN>(args, w, ldsf))
}

// eg_gemm_f32_rows: at most 32 rows of A (a decoded token's projections): reading B
// once from HBM is all such a product costs, so nothing is split over
// workgroups.  A workgroup takes 32 columns; its NW wavefronts take every
// NW-th K step (together 128 NW consecutive bytes of a row), and their sums
// are added in wavefront order.  A wavefront loads a step's 32 rows of B (and
// MR of A) eight lanes to a row's 128 bytes, SETS steps ahead, and turns them
// into fragments (f32_tile's) through 4 + MR / 8 KB of LDS of its own, without
// a barrier: fragments loaded straight from global memory, a lane to a row,
// cost the address path a request a lane (42 us).  131 MB of the PLE key and
// value weights, 5 to 8 rows: 36 us, 32 rows: 44 us; 115 us for gemm_x6_kernel's 256-row tiles
// (196 MB of planes, its parts' sum included).
// The 128 registers of four wavefronts a SIMD are 6 (MR 8) and 16 (MR 32) too few: the
// compiler keeps 28 and 68 bytes a lane in scratch.
constexpr int kFewRows = 32;  // SETS: 2 or 3

template <int NW, int MR, int SETS>
__global__ __launch_bounds__(64 * NW, 4) void gemm_f32_rows_kernel(const F32Args args) {
  constexpr int MA = MR / 8;  // loads of A a step
  // the steps' staging, then the wavefronts' sums
  __shared__ f32x4 lds[NW * 256 > NW * (32 + MR) * 8 ? NW * 256 : NW * (32 + MR) * 8];
  const Plan& p = args.p;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t blocks0 = (p.n[0] + 31) / 32;
  const int grp = (int64_t)blockIdx.x < blocks0 ? 0 : 1;
  const int64_t n0 = 32 * ((int64_t)blockIdx.x - (grp ? blocks0 : 0)), n_grp = p.n[grp];
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  f32x4* mine = lds + wave * (32 + MR) * 8;  // B's 32 rows of 8 chunks, then A's MR
  const int lr = lane >> 3, lc = lane & 7;
  int64_t seg0 = 0;
  for (int s = 0; s < args.n_seg; ++s) {
    const F32Seg& sg = args.seg[s];
    // rows past m or n re-read the last one: not stored
    const float *a[MA], *b[4];
#pragma unroll
    for (int i = 0; i < MA; ++i) a[i] = sg.a + min((int64_t)(lr + 8 * i), p.m - 1) * sg.lda + 4 * lc;
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = sg.b[grp] + min(n0 + lr + 8 * i, n_grp - 1) * sg.ldb[grp] + 4 * lc;
    const int64_t first = (wave - seg0 % NW + NW) % NW, last = sg.ktiles - 1;
    f32x4 fa[SETS][MA], fb[SETS][4];  // sets are named at compile time: registers
    auto load = [&](auto set, int64_t kt) {
      constexpr int f = decltype(set)::value;
      const int64_t k = (kt < last ? kt : last) * kBK;
#pragma unroll
      for (int i = 0; i < 4; ++i) fb[f][i] = *(const f32x4*)(b[i] + k);
#pragma unroll
      for (int i = 0; i < MA; ++i) fa[f][i] = *(const f32x4*)(a[i] + k);
    };
    auto mul = [&](auto set) {
      constexpr int f = decltype(set)::value;
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[(lr + 8 * i) * 8 + swz8(lr + 8 * i, lc)] = fb[f][i];
#pragma unroll
      for (int i = 0; i < MA; ++i) mine[(32 + lr + 8 * i) * 8 + swz8(lr + 8 * i, lc)] = fa[f][i];
      __builtin_amdgcn_wave_barrier();  // a wavefront's LDS accesses run in order
      const int rb = lane & 31, ra = lane & (MR - 1);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int chunk = 4 * (lane >> 5) + c;
        const f32x4 x = mine[(32 + ra) * 8 + swz8(ra, chunk)], y = mine[rb * 8 + swz8(rb, chunk)];
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, acc, 0, 0, 0);
      }
    };
    if (first <= last) {
      constexpr std::integral_constant<int, 0> s0{};
      constexpr std::integral_constant<int, 1> s1{};
      constexpr std::integral_constant<int, SETS - 1> s2{};  // SETS 2: s1 again, unused
      int64_t kt = first;
      auto turn = [&](auto set, int d) {
        mul(set);
        load(set, kt + (d + SETS) * NW);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out here, SETS steps ahead
      };
      load(s0, kt);
      load(s1, kt + NW);
      if constexpr (SETS > 2) load(s2, kt + 2 * NW);
      for (; kt + (SETS - 1) * NW <= last; kt += SETS * NW) {
        turn(s0, 0);
        turn(s1, 1);
        if constexpr (SETS > 2) turn(s2, 2);
      }
      if (kt <= last) mul(s0);
      if (SETS > 2 && kt + NW <= last) mul(s1);
    }
    seg0 += sg.ktiles;
  }
  __syncthreads();
  float* red = (float*)lds;  // [NW][16][64]
#pragma unroll
  for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = acc[r];
  __syncthreads();
  float* out = p.c[grp];
  const int64_t ld = p.ldc[grp];
#pragma unroll
  for (int e = threadIdx.x; e < 1024; e += 64 * NW) {
    const int r = e >> 6, l = e & 63;
    float v = red[r * 64 + l];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[(w * 16 + r) * 64 + l];
    const int64_t row = 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), col = n0 + (l & 31);
    if (row < p.m && col < n_grp) {
      float* q = out + row * ld + col;
      *q = p.accumulate ? *q + v : v;
    }
  }
}

// At most 4 rows of A: on the vector units, where a row of A costs 1 us of
// multiply-adds over those weights (the 32-row MFMA tile costs 16 to 20 us
// whatever it holds).  A wavefront takes 4 columns, 256 k of each at a time
// (a KB of consecutive memory a column), two such steps in flight, and adds
// its lanes' sums at the end; KS 4: the workgroup's wavefronts share 4 columns
// and take every fourth step, for fewer columns than keep the chip's
// wavefronts busy.  One row: 23 us (5.8 TB/s), four: 32 us; 36 us on the
// MFMA kernel.
constexpr int kVecRows = 4, kVecCols = 4;

template <int M, int KS>
__global__ __launch_bounds__(256) void gemm_f32_vec_kernel(const F32Args args) {
  __shared__ float red[4][kVecCols * M];
  const Plan& p = args.p;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t groups0 = (p.n[0] + kVecCols - 1) / kVecCols;
  const int64_t g = KS == 1 ? (int64_t)blockIdx.x * 4 + wave : (int64_t)blockIdx.x;  // column group
  const int grp = g < groups0 ? 0 : 1;
  const int64_t n0 = (g - (grp ? groups0 : 0)) * kVecCols, n_grp = p.n[grp];
  if (n0 >= n_grp) return;  // past the last group (KS 1: no barrier follows)
  float acc[kVecCols][M];
#pragma unroll
  for (int c = 0; c < kVecCols; ++c)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[c][m] = 0.0f;
  for (int s = 0; s < args.n_seg; ++s) {
    const F32Seg& sg = args.seg[s];
    const int64_t k_len = sg.ktiles * kBK;
    const float* b[kVecCols];
#pragma unroll
    for (int c = 0; c < kVecCols; ++c) b[c] = sg.b[grp] + min(n0 + c, n_grp - 1) * sg.ldb[grp];
    f32x4 fa[2][M], fb[2][kVecCols];
    auto load = [&](auto set, int64_t k) {  // a lane past the end multiplies zeros
      constexpr int f = decltype(set)::value;
      const bool in = k < k_len;
      const int64_t kk = in ? k : 0;
#pragma unroll
      for (int c = 0; c < kVecCols; ++c) fb[f][c] = *(const f32x4*)(b[c] + kk);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        fa[f][m] = *(const f32x4*)(sg.a + (m < p.m ? m : 0) * sg.lda + kk);
        if (!in) fa[f][m] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
      }
      if (!in) {
#pragma unroll
        for (int c = 0; c < kVecCols; ++c) fb[f][c] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
      }
    };
    auto mul = [&](auto set) {
      constexpr int f = decltype(set)::value;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < kVecCols; ++c)
#pragma unroll
          for (int m = 0; m < M; ++m) acc[c][m] = fmaf(fa[f][m][e], fb[f][c][e], acc[c][m]);
    };
    constexpr std::integral_constant<int, 0> s0{};
    constexpr std::integral_constant<int, 1> s1{};
    constexpr int STEP = 256 * KS;
    const int64_t base = KS == 1 ? 0 : 256 * wave;  // uniform: the wavefront's first step
    int64_t k = base;
    if (k < k_len) load(s0, k + 4 * lane);
    for (; k + STEP < k_len; k += 2 * STEP) {
      load(s1, k + STEP + 4 * lane);
      mul(s0);
      load(s0, k + 2 * STEP + 4 * lane);
      mul(s1);
    }
    if (k < k_len) mul(s0);
  }
#pragma unroll
  for (int c = 0; c < kVecCols; ++c)
#pragma unroll
    for (int m = 0; m < M; ++m) {
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) acc[c][m] += __shfl_xor(acc[c][m], o);
      if (lane == 0) red[wave][c * M + m] = acc[c][m];
    }
  int e = lane;
  if constexpr (KS > 1) {
    __syncthreads();
    e = threadIdx.x;
  } else {
    __builtin_amdgcn_wave_barrier();  // a wavefront reads its own sums
  }
  if (e >= kVecCols * M) return;
  float v = red[KS == 1 ? wave : 0][e];
#pragma unroll
  for (int w = 1; w < KS; ++w) v += red[w][e];
  const int64_t row = e % M, col = n0 + e / M;
  if (row < p.m && col < n_grp) {
    float* q = p.c[grp] + row * p.ldc[grp] + col;
    *q = p.accumulate ? *q + v : v;
  }
}

// gemm_h3_kernel (eg_gemm_f16x3): fp32 accuracy from three products on the
// fp16 matrix cores; 378 us for the PLE key + value of 2,048 positions, its
// operand's split and gemm_wide_kernel's check included, against 691 us for the
// six bf16 products (bound by the matrix cores and their operands' path
// through LDS, as gemm_x3_kernel).  Every row of an operand's source is scaled by a power of two that
// puts its largest magnitude in [2^14, 2^15) and split into hi = rne16(x) and
// lo = rne16(x - hi): 22 significand bits where the element is at least
// 2^-18 of the row's largest, an absolute 2^-39 of it below.  C = hi*hi +
// hi*lo + lo*hi in fp32, scaled back when it is stored (RowScale); the dropped
// lo*lo is at most 2^-22 of |a||b|.  Half the matrix work of the six bf16
// products (gemm_x6_kernel) and four planes loaded in place of its eight, and
// fewer fp32 additions: its error against float64 is no larger (2048 x 10240 x
// 2560 of N(0, 1): 5.3e-7 in the 2-norm, against 8.3e-7 for the six products
// and for gemm_f32_kernel).  What the planes
// do not hold (values far below their row's largest, an infinity, a NaN) the split
// marks, and gemm_wide_kernel computes the outputs for which it counts.
//
// Planes are fragment-major: 32 rows x 32 k are one 4 KB run, [k half of 16]
// [hi, lo][lane][8 values], lane l holding row l % 32 and k 8 (l / 32) .. + 7 of
// its half: what one MFMA operand register set takes.  A direct-to-LDS load
// then moves 1 KB of consecutive memory (eight whole lines, where the row-major
// planes gave sixteen half lines), a fragment read is 64 consecutive 16-byte
// slots (no bank conflicts, no swizzle), and the load addresses are scalar
// but for the lane's 16 bytes.
//
// Two sources have an exponent each: one source's values far below the
// other's meet products of their own size where B's sources differ the other
// way, so both keep all their bits (with one exponent a row, sources 2^24 apart
// left an error of 4e-5).  A tile (or its part of K) that began in source 0 is
// multiplied by the powers of two that lead to source 1's units when it leaves
// it, in the accumulators, between two steps of the pipeline; kApart bounds them.
// d_emb of 1,531 positions, K 10,240 + 2,560: 247 us (257 us with the pipeline started
// again for source 1).
struct H3Seg {
  const char* a;
  const char* b[2];       // per column group
  int64_t a_blk;          // bytes of one 32-row block (its K steps x 4 KB), both operands
  int64_t a_blocks, b_blocks[2];
  int64_t ktiles;         // K / 32
};

struct H3Args {
  H3Seg seg[1];
  int n_seg;
  Plan p;
  RowScale scale;         // of the last source: the units sums are kept in
  RowScale first;         // of source 0, where there are two
  int64_t kt_first;       // K steps of source 0 where there are two, otherwise all
};

constexpr int kFragBytes = 1024;  // one operand fragment, 64 lanes x 8 fp16
constexpr int kStepBytes = 4 * kFragBytes;  // 32 rows x 32 k, both planes

// The steps of x3_tile (its software pipeline and barriers) over
// fragment-major fp16 planes.
template <int BM, int BN, int WMW, int WNW, bool TWO>
__device__ inline void h3_tile(const H3Args& args, const Work& w, char* lds) {
  constexpr int NW = WMW * WNW, TI = BM / WMW / 32, TJ = BN / WNW / 32;
  constexpr int AB = BM / 32, BB = BN / 32;          // 32-row blocks of a stage
  constexpr int LPW = 4 * (AB + BB) / NW;            // 1 KB loads per wavefront per stage
  constexpr int STAGE = (AB + BB) * kStepBytes;
  static_assert((AB + BB) % NW == 0, "whole blocks per wavefront");
  const Plan& p = args.p;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  const int wm = uwave / WNW, wn = uwave % WNW;
  const H3Seg& sg = args.seg[0];

  int* diff = (int*)(lds + 2 * STAGE);  // two sources: the powers between them, of rows and columns

  f32x16 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int64_t lo = w.kv0, hi = w.kv1;
  // two sources: the step before which the sums so far go into source 1's units
  // (past the last one where the tile's part ends in source 0), if it began in source 0
  const int64_t mid = TWO && lo < args.kt_first ? min(args.kt_first, hi) : -1;
  if (lo < hi) {
    // this wavefront's loads: blocks uwave LB .. + LB - 1 of the stage (A's, then
    // B's), four 1 KB pieces each.  Blocks past the last re-read the last: their
    // products only reach outputs that are not stored.
    constexpr int LB = LPW / 4;
    const char* src[LB];
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      const int blk = uwave * LB + j;
      const bool is_a = blk < AB;
      const int64_t g = is_a ? w.m0 / 32 + blk : w.n0 / 32 + blk - AB;
      const int64_t last = (is_a ? sg.a_blocks : sg.b_blocks[w.grp]) - 1;
      src[j] = (is_a ? sg.a : sg.b[w.grp]) + (g < last ? g : last) * sg.a_blk;
    }
    const uint32_t lane16 = (uint32_t)lane * 16;
    auto piece = [&](int64_t kt, int j, auto sub) {  // the offset advances the global and the LDS address alike
      __builtin_amdgcn_global_load_lds(
          (const void*)(src[j] + kt * kStepBytes + lane16),
          (__attribute__((address_space(3))) void*)(lds + (kt & 1) * STAGE + (uwave * LB + j) * kStepBytes), 16,
          decltype(sub)::value * kFragBytes, 0);
    };
    auto issue_one = [&](int64_t kt, int q) {
      if ((q & 3) == 0) piece(kt, q >> 2, std::integral_constant<int, 0>{});
      if ((q & 3) == 1) piece(kt, q >> 2, std::integral_constant<int, 1>{});
      if ((q & 3) == 2) piece(kt, q >> 2, std::integral_constant<int, 2>{});
      if ((q & 3) == 3) piece(kt, q >> 2, std::integral_constant<int, 3>{});
    };
    auto issue = [&](int64_t kt) {
#pragma unroll
      for (int j = 0; j < LPW; ++j) issue_one(kt, j);
    };
    f16x8 ah[2][TI], al[2][TI], bh[2][TJ], bl[2][TJ];
    auto read = [&](int f, int64_t kt, int ks) {
      const char* st = lds + (kt & 1) * STAGE + ks * 2 * kFragBytes + lane16;
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        ah[f][i] = *(const f16x8*)(st + (wm * TI + i) * kStepBytes);
        al[f][i] = *(const f16x8*)(st + (wm * TI + i) * kStepBytes + kFragBytes);
      }
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        bh[f][j] = *(const f16x8*)(st + (AB + wn * TJ + j) * kStepBytes);
        bl[f][j] = *(const f16x8*)(st + (AB + wn * TJ + j) * kStepBytes + kFragBytes);
      }
    };
    // pass 0: lo*hi, 1: hi*lo, 2: hi*hi
    auto one = [&](int f, int pass, int i, int j) {
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(pass == 0 ? al[f][i] : ah[f][i],
                                                          pass == 1 ? bl[f][j] : bh[f][j], acc[i][j], 0, 0, 0);
    };
    auto mfma = [&](int f, int pass) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) one(f, pass, i, j);
    };
    // the sums into source 1's units: times the rows' and columns' powers
    auto into_second = [&] {
      int lane_o = lane;  // opaque: addresses hoisted out of the walk's loop spill
      asm volatile("" : "+v"(lane_o));
      int sb[TJ];
#pragma unroll
      for (int j = 0; j < TJ; ++j) sb[j] = diff[BM + (wn * TJ + j) * 32 + (lane_o & 31)];
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          __builtin_amdgcn_sched_barrier(0);
          const int4 sa = *(const int4*)(diff + (wm * TI + i) * 32 + 8 * q + 4 * (lane_o >> 5));
          const int sr[4] = {sa.x, sa.y, sa.z, sa.w};
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j][4 * q + r] = ldexpf(acc[i][j][4 * q + r], sr[r] + sb[j]);
        }
      // the powers are read before the barrier that lets the next tile's in
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    issue(lo);
    if (TWO && mid > 0) {  // rows past m or n take the last one's: not stored
      const int e = (int)threadIdx.x;
      static_assert(NW * 64 == BM + BN, "a row or a column a thread");
      if (e < BM) {
        const int64_t row = min(w.m0 + e, p.m - 1);
        diff[e] = args.first.a[row] - args.scale.a[row];
      } else {
        const int64_t col = min(w.n0 + e - BM, p.n[w.grp] - 1);
        diff[e] = args.first.b[w.grp][col] - args.scale.b[w.grp][col];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // in LDS for the others after the barrier below
    }
    if (lo + 1 < hi) {
      issue(lo + 1);
      wait_vm<LPW>();  // this wavefront's part of the first step is in LDS
    } else {
      wait_vm<0>();
    }
    __builtin_amdgcn_s_barrier();
    read(0, lo, 0);
    for (int64_t kt = lo; kt + 1 < hi; ++kt) {
      if (TWO && kt == mid) into_second();
      mfma(0, 0);
      __builtin_amdgcn_sched_barrier(0);  // the reads stay between the passes
      read(1, kt, 1);
      __builtin_amdgcn_sched_barrier(0);
      mfma(0, 1);
      mfma(0, 2);
      __builtin_amdgcn_sched_barrier(0);
      // step kt + 1 is in LDS and step kt in registers, every wavefront's after the barrier
      wait_vm<0>();
      wait_lgkm0();
      __builtin_amdgcn_s_barrier();
      const bool ld = kt + 2 < hi;
#pragma unroll
      for (int t = 0; t < 3 * TI * TJ; ++t) {
        one(1, t / (TI * TJ), (t % (TI * TJ)) / TJ, t % TJ);
        if (t == TI * TJ - 1) {
          __builtin_amdgcn_sched_barrier(0);
          read(0, kt + 1, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        if ((t + 1) % 2 == 0 && (t + 1) / 2 - 1 < LPW) {
          __builtin_amdgcn_sched_barrier(0);
          if (ld) issue_one(kt + 2, (t + 1) / 2 - 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (TWO && mid == hi - 1) into_second();
    mfma(0, 0);
    read(1, hi - 1, 1);
    mfma(0, 1);
    mfma(0, 2);
#pragma unroll
    for (int pass = 0; pass < 3; ++pass) mfma(1, pass);
    if (TWO && mid == hi) into_second();
    __builtin_amdgcn_s_barrier();  // the ring (and powers) are refilled by the next tile
  }
  store_acc<BM, BN, TI, TJ>(p, w, acc, wm, wn, lane, args.scale);
}

template <int BM, int BN, int WMW, int WNW, bool TWO>
__global__ __launch_bounds__(WMW * WNW * 64) void gemm_h3_kernel(const H3Args args) {
  extern __shared__ __attribute__((aligned(16))) char ldsh[];
  EG_GEMM_WALK((h3_tile<BM, BN, WMW, WNW, TWO>(args, w, ldsh)))
}

// The split of eg_gemm_f16x3's operands (eg_split_f16): exponents, marks and
// fragment-major planes of a matrix given as one or two sources side by side
// along K (each padded with zeros to a multiple of 32).
struct F16Src {
  const float* x;
  int64_t cols, row_stride, col_stride;
};

struct SplitF16Args {
  F16Src src[2];
  int64_t chunks[2];      // 8-value chunks of each source, padding included
  int64_t rows, blk;      // blk: bytes of a 32-row block
  char* planes;
  int32_t* exps[2];       // per source: [rows rounded up to 32]
  int32_t* info[2];       // per source and row: kHard, kLossy and the values near the largest
  int32_t* sum8;          // per 8 rows three: a bit a row hard, lossy in source 0, in source 1; the fewest near values
};

// The planes hold a value to 2^-22 of itself down to 2^-18 of the largest of its
// source's part of the row, and to 2^-39 of that largest below.  A row is hard (all
// its outputs computed in fp32) when a source's largest is not finite or so small
// (below 2^-87) that the scale would leave fp32's range.  It is lossy in a source
// when the octaves that its values there lie below 2^-18, and eight times those below
// 2^-24, come to more than 12/128 of one per nonzero value (one in 16 an octave and a half
// below 2^-18, one in 256 below 2^-26).  Rows with fewer small values are not
// lossy, since random rows have some near zero.
// What a lossy row loses counts where the other row is small at its large
// values and only there: an output of it is computed in fp32 unless enough products are
// of two near values, of 2^-7 of their rows' largest at least.  Of K products n_a +
// n_b - K are, n the near values of either row; from K / 16 on sum |a b| is
// at least K 2^-18 of the largest's product and the loss at most 2^-38 K of it, 2^-20
// of sum |a b|.  (A position where one stream's score is near zero is lossy in the
// key's gradient; its near values are that stream's, and no weight is small at
// all of them.  Computing such rows again, one or two of 1,531, cost the block's
// d_emb 121 us.)
constexpr int kWideLow = 40, kNearShare = 16;
constexpr float kLost = 12.0f;  // in 1/128 octaves
constexpr int kHard = 1 << 30, kLossy = 1 << 29, kNear = kLossy - 1;  // kNear: a row of zeros, all near
// Sources of a row more than 2^kApart apart mark it as well: from source 0's
// units to source 1's is then 2^72 at most for a pair of rows, and sums of
// up to 2^44 and products down to 2^-48 stay in fp32's normal range there.
constexpr int kApart = 36;

// A workgroup of 64 NW threads takes ROWS rows of one 32-row block (ROWS 8:
// rows contiguous in memory, a wavefront covers 8 rows x 8 chunks, 256 bytes a
// row; ROWS 32 with TRANS: columns contiguous, a wavefront covers 32 rows x 2
// chunks, 128-byte runs) and all of K.  PER > 0: a thread's PER chunks stay in
// registers between the row maximum and the split; PER 0: they are read
// again.  Bound by HBM: 4 bytes read and 4 written a value.
template <int ROWS, int NW, int PER, bool TRANS>
__global__ __launch_bounds__(64 * NW) void split_f16_kernel(const SplitF16Args a) {
  constexpr int CPW = 64 / ROWS;  // chunks a wavefront covers
  __shared__ uint32_t s_max[2][NW][ROWS];
  __shared__ float s_tally[2][3][NW][ROWS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane % ROWS, cl = lane / ROWS;
  const int64_t r0 = (int64_t)blockIdx.x * ROWS, row = r0 + r;
  const bool live = row < a.rows;
  const int64_t n_chunks = a.chunks[0] + a.chunks[1];

  // both read once: indexed by a lane's source they are loaded before each of its chunks
  const F16Src src0 = a.src[0], src1 = a.src[1];
  auto load = [&](int64_t c, float* v) {
    const int s = c < a.chunks[0] ? 0 : 1;
    const F16Src src = {s ? src1.x : src0.x, s ? src1.cols : src0.cols, s ? src1.row_stride : src0.row_stride,
                        s ? src1.col_stride : src0.col_stride};
    const int64_t k = (s ? c - a.chunks[0] : c) * 8;
    const float* x = src.x + row * src.row_stride + k * src.col_stride;
    if (!live || c >= n_chunks) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.0f;
    } else if (!TRANS && k + 8 <= src.cols && (src.row_stride & 3) == 0 && ((uintptr_t)src.x & 15) == 0) {
      const float4 p = *(const float4*)x, q = *(const float4*)(x + 4);
      v[0] = p.x, v[1] = p.y, v[2] = p.z, v[3] = p.w;
      v[4] = q.x, v[5] = q.y, v[6] = q.z, v[7] = q.w;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = k + e < src.cols ? x[e * src.col_stride] : 0.0f;
    }
  };
  uint32_t mxs[2] = {0, 0};  // per source
  auto see = [&](int64_t c, const float* v) {
    uint32_t m = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) m = max(m, __float_as_uint(v[e]) & 0x7fffffffu);
    if (c < a.chunks[0]) mxs[0] = max(mxs[0], m);
    else mxs[1] = max(mxs[1], m);
  };
  float kept[PER > 0 ? PER : 1][8];
  if constexpr (PER > 0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) load((int64_t)(i * NW + wave) * CPW + cl, kept[i]);
#pragma unroll
    for (int i = 0; i < PER; ++i) see((int64_t)(i * NW + wave) * CPW + cl, kept[i]);
  } else {
    for (int64_t c = wave * CPW + cl; c < n_chunks; c += 2 * NW * CPW) {
      float v[2][8];
      load(c, v[0]);
      load(c + NW * CPW, v[1]);
      see(c, v[0]);
      see(c + NW * CPW, v[1]);
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int o = 32; o >= ROWS; o >>= 1) mxs[s] = max(mxs[s], (uint32_t)__shfl_xor((int)mxs[s], o));
    if (lane < ROWS) s_max[s][wave][r] = mxs[s];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    mxs[0] = max(mxs[0], s_max[0][q][r]);
    mxs[1] = max(mxs[1], s_max[1][q][r]);
  }
  // out of the scale's range, or the sources too far apart: no planes
  bool out = false;
  int ex[2];
  float scale[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    ex[s] = (int)(mxs[s] >> 23);
    out |= mxs[s] != 0 && (ex[s] >= 255 || ex[s] < kWideLow);
  }
  // a source of zeros takes the other's exponent
  ex[0] = mxs[0] == 0 ? ex[1] : ex[0];
  ex[1] = mxs[1] == 0 ? ex[0] : ex[1];
  out |= abs(ex[0] - ex[1]) > kApart;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    // the source times 2^(14 - e) has its largest magnitude in [2^14, 2^15)
    ex[s] = out || ex[s] == 0 ? 14 : ex[s] - 127;
    scale[s] = __uint_as_float((uint32_t)(127 + 14 - ex[s]) << 23);
  }
  if (wave == 0 && lane < ROWS && live) {
    a.exps[0][row] = ex[0] - 14;
    a.exps[1][row] = ex[1] - 14;
  }
  // per source: nonzero values, near values, and 1/128 octaves lost, from the upper
  // halves of two values a word at a time (8 bits of exponent, 7 of the significand).
  // 1,531 rows of 12,800 values: 69 us, 64 us with the planes and one count alone
  float tally[2][3] = {};
  u16x2 one = 1;
  asm("" : "+v"(one));  // min(h, 1) stays that: two compares and selects a word otherwise
  auto put = [&](int64_t c, const float* v) {
    if (c >= n_chunks) return;
    f16x8 hi, lo;
    const int s = c < a.chunks[0] ? 0 : 1;
    const float sc = s ? scale[1] : scale[0];
    const uint16_t t18 = (uint16_t)(((s ? mxs[1] : mxs[0]) >> 16) - 18 * 128);  // above 24 octaves' unless out or zero
    const u16x2 v18 = t18, v24 = (uint16_t)(t18 - 6 * 128), v7 = (uint16_t)(t18 + 11 * 128 - 1);
    uint32_t seen = 0, lost = 0, pair = 0;  // seen: nonzero + 256 near
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float y = v[e];
      asm("" : "+v"(y));  // nothing of the maximum's pass is kept in registers for this one
      if (e & 1) {
        const uint32_t tops = __builtin_amdgcn_perm(__float_as_uint(y), pair, 0x07060302) & 0x7fff7fffu;
        const u16x2 h = __builtin_bit_cast(u16x2, tops), z = h - one;  // zero wraps to the largest
        lost = __builtin_amdgcn_udot2(__builtin_elementwise_sub_sat(v18, z), one, lost, false);
        lost = __builtin_amdgcn_udot2(__builtin_elementwise_sub_sat(v24, z), (u16x2)8, lost, false);
        seen = __builtin_amdgcn_udot2(__builtin_elementwise_min(h, one), one, seen, false);
        seen = __builtin_amdgcn_udot2(__builtin_elementwise_min(__builtin_elementwise_sub_sat(h, v7), one),
                                      (u16x2)256, seen, false);
      }
      pair = __float_as_uint(y);
      const float x = out ? 0.0f : y * sc;
      hi[e] = (_Float16)x;
      lo[e] = (_Float16)(x - (float)hi[e]);
    }
    const float got[3] = {(float)(seen & 0xff), (float)(seen >> 8), (float)lost};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      tally[0][q] += s ? 0.0f : got[q];
      tally[1][q] += s ? got[q] : 0.0f;
    }
    char* o = a.planes + (row >> 5) * a.blk + (c >> 2) * kStepBytes + ((c >> 1) & 1) * 2 * kFragBytes +
              ((row & 31) + 32 * (c & 1)) * 16;
    *(f16x8*)o = hi;
    *(f16x8*)(o + kFragBytes) = lo;
  };
  if constexpr (PER > 0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      put((int64_t)(i * NW + wave) * CPW + cl, kept[i]);
      __builtin_amdgcn_sched_barrier(0);  // one chunk's values at a time: several at once take 80 registers more
    }
  } else {
    for (int64_t c = wave * CPW + cl; c < n_chunks; c += 2 * NW * CPW) {
      float v[2][8];
      load(c, v[0]);
      load(c + NW * CPW, v[1]);
      put(c, v[0]);
      put(c + NW * CPW, v[1]);
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int o = 32; o >= ROWS; o >>= 1) tally[s][q] += __shfl_xor(tally[s][q], o);
      if (lane < ROWS) s_tally[s][q][wave][r] = tally[s][q];
    }
  __syncthreads();
  if (wave != 0) return;
  // lanes of the same row hold the same
  int fewest[2];
  uint64_t lossy[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      tally[s][q] = 0.0f;
#pragma unroll
      for (int u = 0; u < NW; ++u) tally[s][q] += s_tally[s][q][u][r];
    }
    const bool is = tally[s][2] > kLost * tally[s][0];
    fewest[s] = tally[s][0] == 0.0f || !live ? kNear : (int)fminf(tally[s][1], (float)(kNear / 2));
    if (lane < ROWS && live) a.info[s][row] = fewest[s] | (is ? kLossy : 0) | (out ? kHard : 0);
    lossy[s] = __ballot(is);
#pragma unroll
    for (int o = 4; o >= 1; o >>= 1) fewest[s] = min(fewest[s], __shfl_xor(fewest[s], o));
    fewest[s] = __shfl(fewest[s], 8 * lane & 63);  // of rows 8 lane .. 8 lane + 7
  }
  const uint64_t hard = __ballot(out);
  if (lane < ROWS / 8 && r0 + 8 * lane < a.rows) {
    int32_t* o = a.sum8 + 3 * (r0 / 8 + lane);
    o[0] = (int32_t)((hard >> 8 * lane & 0xff) | (lossy[0] >> 8 * lane & 0xff) << 8 |
                     (lossy[1] >> 8 * lane & 0xff) << 16);
    o[1] = fewest[0];
    o[2] = fewest[1];
  }
}

// The outputs that the planes do not give (hard rows; lossy rows against rows with too few near
// values), in fp32: a 32 x 32 tile that has one is computed again from the fp32 operands
// (any strides) on the fp32 matrix cores, and those outputs are stored: an output
// depends on its own two rows alone.  There are few such rows, and then only their
// strip of tiles is there to do, so the eight wavefronts of a workgroup share a
// tile, each taking every eighth 32 k of it straight into registers (the next
// step's while one is multiplied, no barrier), and their sums are added in
// wavefront order; a step whose part of A is all zeros (positions without a
// loss, in a weight gradient) is skipped.  Without such a row a workgroup
// reads the marks of its tiles and ends (5 us).  One hard row: d_emb of 2,560
// columns and K 12,800 121 us, bound by its 80 tiles' loads and the fp32 matrix
// cores of 80 CUs; 12,800 columns, K 2,560 57 us (64 x 64 tiles through LDS 200
// and 108 us; 4 and 16 wavefronts 148 and 128 us).  Every row, 12,800 x
// 2,560 outputs, K 1,531: 1.7 ms, bound by the 12.5 GB its tiles read from L2
// (1.3 ms on 64 x 64 tiles, 5.8 ms on the vector units).
constexpr int kWideGroups = 509;  // two workgroups a CU, and prime, so that a row's strip of
                                  // tiles and a column's go over all of them
constexpr int kWideWaves = 8;

struct WideArgs {
  F16Src a[2], b[2][2];    // sources of A and of B per column group
  const int32_t* info[3][2];  // of A, B, B2
  const int32_t* sum8[3];
  int near[2];             // near values of two rows together from which their output stays, per source
  int n_src;
  int64_t m, n[2];
  float* c[2];
  int64_t ldc[2];
};

__global__ __launch_bounds__(64 * kWideWaves, 4) void gemm_wide_kernel(const WideArgs g) {
  constexpr int NT = 64 * kWideWaves;
  __shared__ float s_part[kWideWaves][16][64];
  __shared__ int s_tile[NT], s_info[2][2][32];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
  const int64_t tm_n = (g.m + 31) / 32, tn0 = (g.n[0] + 31) / 32, tn_n = tn0 + (g.n[1] + 31) / 32;
  const int64_t pitch = tn_n % kWideGroups == 0 ? tn_n + 1 : tn_n, tiles = tm_n * pitch;
  // of an output's row and column, or of a tile's two sides: their marks, and near values together
  auto needed = [&](int hard, int lossy0, int lossy1, int n0, int n1) {
    return hard != 0 || (lossy0 != 0 && n0 < g.near[0]) || (lossy1 != 0 && n1 < g.near[1]);
  };
  // of the 32 rows of a side's tile: their marks, and the fewest near values
  auto side = [&](int x, int64_t t, int64_t rows, int* n) {
    int mark = 0;
    n[0] = n[1] = kNear;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t* o = g.sum8[x] + 3 * (4 * t + q);
      if (32 * t + 8 * q < rows) mark |= o[0], n[0] = min(n[0], o[1]), n[1] = min(n[1], o[2]);
    }
    return mark;
  };
  // NT of the workgroup's tiles at a time: those with outputs to compute, in order
  for (int64_t base = blockIdx.x; base < tiles; base += (int64_t)kWideGroups * NT) {
    const int64_t mine = base + (int64_t)kWideGroups * tid;
    int mark = 0;
    if (mine < tiles && mine % pitch < tn_n) {
      const int64_t tn = mine % pitch;
      const int grp = tn < tn0 ? 0 : 1;
      int na[2], nb[2];
      const int both = side(0, mine / pitch, g.m, na) | side(1 + grp, grp ? tn - tn0 : tn, g.n[grp], nb);
      mark = needed(both & 0xff, both >> 8 & 0xff, both >> 16 & 0xff, na[0] + nb[0], na[1] + nb[1]);
    }
    if (!__syncthreads_or(mark)) continue;
    s_tile[tid] = mark != 0;
    __syncthreads();
    for (int64_t i = 0; i < NT && base + kWideGroups * i < tiles; ++i) {
      if (!s_tile[i]) continue;  // the same for every thread
      const int64_t tile = base + kWideGroups * i, tm = tile / pitch, tn = tile % pitch;
      const int grp = tn < tn0 ? 0 : 1;
      const int64_t m0 = 32 * tm, n0 = 32 * (grp ? tn - tn0 : tn), n_grp = g.n[grp];
      if (tid < 128) {  // rows past the end take the last one's: not stored
        const int x = tid >> 6 ? 1 + grp : 0, s = tid >> 5 & 1;
        s_info[tid >> 6][s][tid & 31] = g.info[x][s][min((x ? n0 : m0) + (tid & 31), (x ? n_grp : g.m) - 1)];
      }
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
      for (int s = 0; s < g.n_src; ++s) {
        const F16Src &xa = g.a[s], &xb = g.b[grp][s];
        const int64_t k_len = xa.cols;
        // a lane's row (past the end the last one: not stored) and, of 32 k, its half's sixteen
        const float* pa = xa.x + min(m0 + (lane & 31), g.m - 1) * xa.row_stride + 16 * half * xa.col_stride;
        const float* pb = xb.x + min(n0 + (lane & 31), n_grp - 1) * xb.row_stride + 16 * half * xb.col_stride;
        auto load = [&](const F16Src& x, const float* p, int64_t k, float* v) {
          p += k * x.col_stride;
          if (k + 32 > k_len) {  // the last step: zeros past the end
            const int left = (int)(k_len - k) - 16 * half;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              v[e] = e < left ? *p : 0.0f;
              p += x.col_stride;
              asm volatile("" : "+v"(p));  // one address at a time: sixteen of them spill
            }
          } else if (x.col_stride == 1 && (x.row_stride & 3) == 0 && ((uintptr_t)x.x & 15) == 0) {
#pragma unroll
            for (int e = 0; e < 16; e += 4) {
              const f32x4 y = *(const f32x4*)(p + e);
              v[e] = y.x, v[e + 1] = y.y, v[e + 2] = y.z, v[e + 3] = y.w;
            }
          } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              v[e] = *p;
              p += x.col_stride;
              asm volatile("" : "+v"(p));
            }
          }
        };
        float na[16], nb[16];
        int64_t k = 32 * __builtin_amdgcn_readfirstlane(wave);
        if (k < k_len) {
          load(xa, pa, k, na);
          load(xb, pb, k, nb);
        }
#pragma unroll 1
        for (; k < k_len; k += 32 * kWideWaves) {
          float fa[16], fb[16];
          bool some = false;  // a value of A, or one of B whose product with zero is not zero
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            fa[e] = na[e], fb[e] = nb[e];
            some |= fa[e] != 0.0f || (__float_as_uint(fb[e]) & 0x7f800000u) == 0x7f800000u;
          }
          if (k + 32 * kWideWaves < k_len) {
            load(xa, pa, k + 32 * kWideWaves, na);
            load(xb, pb, k + 32 * kWideWaves, nb);
          }
          if (__ballot(some) == 0) continue;
#pragma unroll
          for (int e = 0; e < 16; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s_part[wave][r][lane] = acc[r];
      __syncthreads();
#pragma unroll
      for (int r = wave; r < 16; r += kWideWaves) {
        const int lr = 8 * (r >> 2) + 4 * half + (r & 3), lc = lane & 31;
        float v = s_part[0][r][lane];
#pragma unroll
        for (int w = 1; w < kWideWaves; ++w) v += s_part[w][r][lane];
        const int a0 = s_info[0][0][lr], a1 = s_info[0][1][lr], b0 = s_info[1][0][lc], b1 = s_info[1][1][lc];
        const bool marked = needed((a0 | b0) & kHard, (a0 | b0) & kLossy, (a1 | b1) & kLossy,
                                   (a0 & kNear) + (b0 & kNear), (a1 & kNear) + (b1 & kNear));
        if (marked && m0 + lr < g.m && n0 + lc < n_grp) g.c[grp][(m0 + lr) * g.ldc[grp] + n0 + lc] = v;
      }
      __syncthreads();  // the sums and marks are read
    }
  }
}

// C (+)= the sum of a last-round tile's pieces, in K order: BM BN / 1024
// blocks a tile, each thread four consecutive columns of one row.
template <int BM, int BN, typename Scale>
__global__ __launch_bounds__(256) void piece_sum_kernel(const Plan p, const Scale scale) {
  constexpr int kBlocks = BM * BN / 1024;
  const int q = blockIdx.x / kBlocks;
  const int e = (blockIdx.x % kBlocks) * 256 + threadIdx.x;  // float4 of the BM x BN tile
  const int lr = e / (BN / 4), lc = (e % (BN / 4)) * 4;
  int tm, tn;
  grouped(p.dp_tiles + q, p.tiles_m, p.tiles_n, tm, tn);
  const int grp = tn < p.tiles_n0 ? 0 : 1;
  const int64_t row = (int64_t)tm * BM + lr;
  if (row >= p.m) return;
  const float4* ws = (const float4*)(p.ws + (int64_t)q * p.pieces * (BM * BN)) + e;
  float4 v = ws[0];
  for (int s = 1; s < p.pieces; ++s) {
    const float4 u = ws[(int64_t)s * (BM * BN / 4)];
    v.x += u.x;
    v.y += u.y;
    v.z += u.z;
    v.w += u.w;
  }
  const int64_t n_grp = p.n[grp], col0 = (int64_t)(grp ? tn - p.tiles_n0 : tn) * BN + lc;
  float* out = p.c[grp] + row * p.ldc[grp];
  const float vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int64_t col = col0 + t;
    if (col < n_grp) {
      const float x = scale(vv[t], grp, row, col);
      out[col] = p.accumulate ? out[col] + x : x;
    }
  }
}

// C (+)= the sum, in K order, of the parts of a last-round tile that the
// ranges computed: the ranges meeting the tile, in increasing order (a tile
// one range covers whole was stored directly).  A range holds at least 8
// units, so the tile's parts are those of the consecutive ranges s0 .. s1, and
// only s0 can have begun in an earlier tile.  A thread sums kSumRows float4,
// one row of four apart, all their loads of a part in flight, and stores four
// columns at once where C allows it: bound by HBM (the parts and C).  On the
// PLE key + value of 2,048 positions (100 MB of parts, 38 MB of C) 24 us,
// 41 us with one float4 and the ranges' 64-bit divisions a thread.
constexpr int kSumRows = 4;

template <int BM, int BN, typename Scale>
__global__ __launch_bounds__(256) void sk_sum_kernel(const Plan p, const Scale scale) {
  constexpr int kBlocks = BM * BN / 1024 / kSumRows;
  constexpr int kRowsApart = 1024 / BN;  // rows of the tile 256 threads of float4 cover
  const int q = blockIdx.x / kBlocks;    // last-round tile
  const int lr0 = (int)(blockIdx.x % kBlocks) * kSumRows * kRowsApart + (int)threadIdx.x / (BN / 4);
  const int lc = ((int)threadIdx.x % (BN / 4)) * 4;
  const int64_t kt = p.kt_total, x0 = (int64_t)q * kt, x1 = x0 + kt;
  // the last s with start(s) <= x: floor(U s / G) <= x  <=>  U s < (x + 1) G
  const int64_t s0 = ((x0 + 1) * p.sk_groups - 1) / p.sk_units, s1 = (x1 * p.sk_groups - 1) / p.sk_units;
  if (s0 == s1) return;  // one range covers the tile: stored directly
  int tm, tn;
  grouped(p.dp_tiles + q, p.tiles_m, p.tiles_n, tm, tn);
  const int grp = tn < p.tiles_n0 ? 0 : 1;
  const float* ws = p.ws + lr0 * BN + lc;
  const int64_t first = 2 * s0 + (sk_start(p, s0) < x0 ? 1 : 0);
  float4 v[kSumRows];
#pragma unroll
  for (int r = 0; r < kSumRows; ++r) v[r] = *(const float4*)(ws + first * (BM * BN) + r * kRowsApart * BN);
  for (int64_t s = s0 + 1; s <= s1; ++s) {
#pragma unroll
    for (int r = 0; r < kSumRows; ++r) {
      const float4 u = *(const float4*)(ws + 2 * s * (BM * BN) + r * kRowsApart * BN);
      v[r].x += u.x;
      v[r].y += u.y;
      v[r].z += u.z;
      v[r].w += u.w;
    }
  }
  const int64_t n_grp = p.n[grp], col0 = (int64_t)(grp ? tn - p.tiles_n0 : tn) * BN + lc, ld = p.ldc[grp];
  const bool whole = col0 + 4 <= n_grp && (ld & 3) == 0 && ((uintptr_t)p.c[grp] & 15) == 0 && !p.accumulate;
#pragma unroll
  for (int r = 0; r < kSumRows; ++r) {
    const int64_t row = (int64_t)tm * BM + lr0 + r * kRowsApart;
    if (row >= p.m) return;
    float* out = p.c[grp] + row * ld;
    const float vv[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
    if (whole) {
      *(float4*)(out + col0) = make_float4(scale(vv[0], grp, row, col0), scale(vv[1], grp, row, col0 + 1),
                                           scale(vv[2], grp, row, col0 + 2), scale(vv[3], grp, row, col0 + 3));
      continue;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int64_t col = col0 + t;
      if (col < n_grp) {
        const float x = scale(vv[t], grp, row, col);
        out[col] = p.accumulate ? out[col] + x : x;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Host side

struct PiecePlan {
  int dp;              // whole tiles
  int pieces;          // pieces per remaining tile
  int64_t kt_per_piece;
  int sk_groups;       // > 0: the remaining tiles' K steps in this many contiguous ranges instead of pieces
};

// A kernel's tile: BM x BN outputs of `threads` threads and `lds` bytes of
// LDS.  The plan counts `rounds_per_cu` tiles a CU as one round (one for
// both kernels' 256 x 256 tiles, whose LDS holds one workgroup a CU).
// `sum_cost` / (K steps) is the time of summing one round of pieces against
// the time of one round of tiles: 4 bytes read per output and piece at ~5
// TB/s against 192 (bf16 products, ~1 PFLOP/s reached) or 64 (fp32, ~130
// TFLOP/s) flops per output and K step.
// `ranges`: the kernel can take the last round as contiguous K ranges, one per
// workgroup of the round (gemm_f32_kernel), rather than as equal pieces of each
// tile.
struct Shape {
  int bm, bn, threads, rounds_per_cu;
  size_t lds;
  double sum_cost;
  bool ranges;
};

constexpr Shape kX3Shape{kX3BM, kX3BN, kX3WM * kX3WN * 64, 1, (size_t)kStages * 2 * (kX3BM + kX3BN) * kBK * 2, 4.2,
                         true};
constexpr Shape kH3TwoShape{kX3BM, kX3BN, kX3WM * kX3WN * 64, 1, kX3Shape.lds + (kX3BM + kX3BN) * 4, 4.2, true};
constexpr int kF32BM = 256, kF32BN = 256;
constexpr Shape kF32Shape{kF32BM, kF32BN, kF32BM * kF32BN / 64, 1,
                          (size_t)kStages * (kF32BM + kF32BN) * kBK * 4, 1.6, true};

// k_slices >= 1: every tile in k_slices pieces (1: whole tiles).  0: the
// tiles of a partly filled last round (of `slots` tiles) in the piece count
// that minimises the time of that round in tile units, ceil(R s / slots) / s,
// plus the cost of summing the pieces, sum_cost / (K steps) per round of
// pieces.  At least 8 K steps a piece, and only for a gain of 10 % or more.
PiecePlan plan_pieces(int64_t tiles, int64_t kt_total, int k_slices, int slots, double sum_cost) {
  PiecePlan pp{(int)tiles, 1, kt_total > 0 ? kt_total : 1, 0};
  int s = 1;
  if (k_slices >= 1) {
    s = k_slices;
  } else {
    const int64_t r = tiles % slots;
    if (r == 0 || kt_total < 16) return pp;
    const double per_round = sum_cost / (double)kt_total;
    double best = 1.0;
    for (int c = 2; c <= 8 && kt_total / c >= 8; ++c) {
      const double t = (double)((r * c + slots - 1) / slots) / c + per_round * (double)(r * c) / slots;
      if (t < best) {
        best = t;
        s = c;
      }
    }
    if (best > 0.9) return pp;
  }
  if (kt_total < s) s = kt_total > 0 ? (int)kt_total : 1;
  if (s <= 1) return pp;
  pp.kt_per_piece = (kt_total + s - 1) / s;
  pp.pieces = (int)((kt_total + pp.kt_per_piece - 1) / pp.kt_per_piece);
  if (pp.pieces <= 1) {
    pp.pieces = 1;
    pp.kt_per_piece = kt_total;
    return pp;
  }
  pp.dp = k_slices >= 1 ? 0 : (int)(tiles - tiles % slots);
  return pp;
}

// CUs of the current device.
int device_cus(int* cus_out) {
  static std::mutex mu;
  static std::vector<std::pair<int, int>> known;  // (device, CU count)
  int dev = 0;
  EG_CHECK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  for (const auto& k : known)
    if (k.first == dev) {
      *cus_out = k.second;
      return EG_OK;
    }
  int cus = 0;
  EG_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  EG_CHECK_ARG(cus > 0, "device %d reports %d CUs", dev, cus);
  known.emplace_back(dev, cus);
  *cus_out = cus;
  return EG_OK;
}

int64_t tiles_of(const Shape& sh, int64_t m, int64_t n, int64_t n2) {
  return ((m + sh.bm - 1) / sh.bm) * ((n + sh.bn - 1) / sh.bn + (n2 + sh.bn - 1) / sh.bn);
}

int64_t piece_bytes(const Shape& sh, int64_t tiles, const PiecePlan& pp) {
  const int64_t tile = (int64_t)sh.bm * sh.bn * (int64_t)sizeof(float);
  if (pp.sk_groups > 0) return 2 * (int64_t)pp.sk_groups * tile;
  return pp.pieces > 1 ? (tiles - pp.dp) * pp.pieces * tile : 0;
}

int plan_for(const Shape& sh, int64_t m, int64_t n, int64_t n2, int64_t kt_total, int k_slices, int64_t* tiles,
             PiecePlan* pp) {
  int cus = 0;
  const int rc = device_cus(&cus);
  if (rc != EG_OK) return rc;
  *tiles = tiles_of(sh, m, n, n2);
  const int slots = sh.rounds_per_cu * cus;
  *pp = plan_pieces(*tiles, kt_total, k_slices, slots, sh.sum_cost);
  // a kernel that takes ranges: the last round that the plan cuts runs as one
  // contiguous range of its (tile, K step) units per workgroup slot, at least
  // 8 K steps a range (fewer pieces than equal cuts, and no tile cut more
  // often than the ranges meeting it)
  const int64_t r = *tiles - pp->dp;
  if (sh.ranges && k_slices == 0 && pp->pieces > 1 && r < slots && r * kt_total >= 8 * (int64_t)slots) {
    pp->pieces = 1;
    pp->kt_per_piece = kt_total;
    pp->sk_groups = slots;
  }
  return EG_OK;
}

int64_t workspace_size(const Shape& sh, int64_t m, int64_t n, int64_t n2, int64_t k, int32_t k_slices) {
  if (m <= 0 || n < 0 || n2 < 0 || n + n2 == 0 || k < 0 || k_slices < 0) return 0;
  int64_t tiles = 0;
  PiecePlan pp{};
  if (plan_for(sh, m, n, n2, k / 32, k_slices, &tiles, &pp) != EG_OK) return -1;
  return piece_bytes(sh, tiles, pp);
}

// The part of both entry points after their operands are checked: the plan,
// the LDS attribute, the launch and the pieces' sum.
template <int BM, int BN, typename Args, typename Scale = NoScale>
int launch_gemm(const Shape& sh, void (*kernel)(const Args), const char* name, Args& g, int64_t m, int64_t n,
                int64_t n2, float* c, int64_t ldc, float* c2, int64_t ldc2, int32_t accumulate, int32_t k_slices,
                void* workspace, int64_t workspace_bytes, void* stream, const Scale& scale = Scale{}) {
  EG_CHECK_ARG(m >= 0 && n >= 0 && n2 >= 0 && k_slices >= 0, "m=%lld n=%lld n2=%lld k_slices=%d", (long long)m,
               (long long)n, (long long)n2, k_slices);
  EG_CHECK_ARG(n == 0 || (c != nullptr && ldc >= n), "c / ldc");
  EG_CHECK_ARG(n2 == 0 || (c2 != nullptr && ldc2 >= n2), "c2 / ldc2");
  if (m == 0 || n + n2 == 0) return 0;
  Plan& p = g.p;
  p.kt0 = g.n_seg > 0 ? g.seg[0].ktiles : 0;
  p.kt_total = p.kt0;
  for (int s = 1; s < g.n_seg; ++s) p.kt_total += g.seg[s].ktiles;
  int64_t tiles = 0;
  PiecePlan pp{};
  int rc = plan_for(sh, m, n, n2, p.kt_total, k_slices, &tiles, &pp);
  if (rc != EG_OK) return rc;
  EG_CHECK_ARG(tiles < (1LL << 24), "too many tiles");
  const int64_t need = piece_bytes(sh, tiles, pp);
  if (need > 0) {
    EG_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace & 15) == 0 && workspace_bytes >= need,
                 "this call needs a 16-byte aligned workspace of %lld bytes (its _workspace_size function)",
                 (long long)need);
    p.ws = (float*)workspace;
  }
  p.dp_tiles = pp.dp;
  p.pieces = pp.pieces;
  p.kt_per_piece = pp.kt_per_piece;
  p.sk_groups = pp.sk_groups;
  p.sk_units = pp.sk_groups > 0 ? (tiles - pp.dp) * p.kt_total : 0;
  p.c[0] = c;
  p.c[1] = c2;
  p.ldc[0] = ldc;
  p.ldc[1] = ldc2;
  p.m = m;
  p.n[0] = n;
  p.n[1] = n2;
  p.tiles_m = (int)((m + BM - 1) / BM);
  p.tiles_n0 = (int)((n + BN - 1) / BN);
  p.tiles_n = p.tiles_n0 + (int)((n2 + BN - 1) / BN);
  p.accumulate = accumulate ? 1 : 0;
  const int64_t blocks = pp.dp + (pp.sk_groups > 0 ? (int64_t)pp.sk_groups : (tiles - pp.dp) * pp.pieces);
  EG_CHECK_ARG(blocks < (1LL << 31), "too many workgroups");
  hipStream_t st = (hipStream_t)stream;
  // the dynamic LDS attribute, once per device and kernel
  static std::mutex mu;
  static std::vector<std::pair<const void*, int>> done;
  int dev = 0;
  EG_CHECK_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lock(mu);
    const std::pair<const void*, int> key((const void*)kernel, dev);
    if (std::find(done.begin(), done.end(), key) == done.end()) {
      EG_CHECK_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)sh.lds));
      done.push_back(key);
    }
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(sh.threads), sh.lds, st, g);
  rc = launch_status(name);
  if (rc != 0 || pp.dp == tiles) return rc;
  const dim3 sum_grid((unsigned)((tiles - pp.dp) * (BM * BN / 1024)));
  if (pp.sk_groups > 0) {
    hipLaunchKernelGGL((sk_sum_kernel<BM, BN, Scale>), dim3(sum_grid.x / kSumRows), dim3(256), 0, st, p, scale);
    return launch_status("sk_sum_kernel");
  }
  hipLaunchKernelGGL((piece_sum_kernel<BM, BN, Scale>), sum_grid, dim3(256), 0, st, p, scale);
  return launch_status("piece_sum_kernel");
}

}  // namespace
}  // namespace eg

extern "C" {

}  // extern "C"

namespace eg {
namespace {
// eg_split_bf16 (lo2 == nullptr) and eg_split_bf16x6.
int split_planes(const float* x, int64_t rows, int64_t cols, int64_t ld, void* hi, void* lo, void* lo2,
                 void* stream) {
  EG_CHECK_ARG(rows >= 0 && cols >= 0 && ld >= cols, "rows=%lld cols=%lld ld=%lld", (long long)rows, (long long)cols,
               (long long)ld);
  const int64_t kp = (cols + 31) / 32 * 32;
  if (rows == 0 || kp == 0) return 0;
  EG_CHECK_ARG(x != nullptr && hi != nullptr && lo != nullptr, "NULL argument");
  EG_CHECK_ARG(((uintptr_t)hi & 15) == 0 && ((uintptr_t)lo & 15) == 0 && ((uintptr_t)lo2 & 15) == 0,
               "the planes must be 16-byte aligned");
  const dim3 grid((unsigned)((kp / 4 + 255) / 256), (unsigned)(rows < 65535 ? rows : 65535));
  const bool vec = ld % 4 == 0 && ((uintptr_t)x & 15) == 0;
  hipStream_t st = (hipStream_t)stream;
  __bf16 *h = (__bf16*)hi, *l = (__bf16*)lo, *l2 = (__bf16*)lo2;
  if (lo2 != nullptr) {
    if (vec) hipLaunchKernelGGL((split_kernel<true, true>), grid, dim3(256), 0, st, x, rows, cols, ld, kp, h, l, l2);
    else hipLaunchKernelGGL((split_kernel<false, true>), grid, dim3(256), 0, st, x, rows, cols, ld, kp, h, l, l2);
  } else {
    if (vec) hipLaunchKernelGGL((split_kernel<true, false>), grid, dim3(256), 0, st, x, rows, cols, ld, kp, h, l, l2);
    else hipLaunchKernelGGL((split_kernel<false, false>), grid, dim3(256), 0, st, x, rows, cols, ld, kp, h, l, l2);
  }
  return launch_status("split_kernel");
}
}  // namespace
}  // namespace eg

extern "C" {

int eg_split_bf16(const float* x, int64_t rows, int64_t cols, int64_t ld, void* hi, void* lo, void* stream) {
  return eg::split_planes(x, rows, cols, ld, hi, lo, nullptr, stream);
}

int eg_split_bf16x6(const float* x, int64_t rows, int64_t cols, int64_t ld, void* hi, void* mid, void* lo,
                    void* stream) {
  EG_CHECK_ARG(lo != nullptr, "NULL argument");
  return eg::split_planes(x, rows, cols, ld, hi, mid, lo, stream);
}

int64_t eg_gemm_workspace_size(int64_t m, int64_t n, int64_t n2, int64_t k, int32_t k_slices) {
  return eg::workspace_size(eg::kX3Shape, m, n, n2, k, k_slices);
}

int64_t eg_gemm_f32_workspace_size(int64_t m, int64_t n, int64_t n2, int64_t k, int32_t k_slices) {
  return eg::workspace_size(eg::kF32Shape, m, n, n2, k, k_slices);
}

}  // extern "C"

namespace eg {
namespace {
// The kernel arguments of eg_gemm_bf16x3 / eg_gemm_bf16x6 operands (the planes checked).
int bf16_operands(const eg_gemm_operands* ops, int32_t n_seg, int64_t m, int64_t n, int64_t n2, GemmArgs& g) {
  EG_CHECK_ARG(ops != nullptr && n_seg >= 0 && n_seg <= 2, "n_seg=%d", n_seg);
  for (int s = 0; s < n_seg; ++s) {
    const eg_gemm_operands& o = ops[s];
    EG_CHECK_ARG(o.k >= 0 && o.k % 32 == 0, "segment %d: k must be a multiple of 32 (k=%lld)", s, (long long)o.k);
    if (o.k == 0) continue;
    const void* planes[6] = {o.a_hi, o.a_lo, o.b_hi, o.b_lo, o.b2_hi, o.b2_lo};
    for (int q = 0; q < 6; ++q) {
      if (q >= 4 && n2 == 0) break;
      EG_CHECK_ARG(planes[q] != nullptr && ((uintptr_t)planes[q] & 15) == 0,
                   "segment %d: plane %d is NULL or not 16-byte aligned", s, q);
    }
    EG_CHECK_ARG(o.lda % 8 == 0 && o.ldb % 8 == 0 && o.lda >= o.k && o.ldb >= o.k &&
                     (n2 == 0 || (o.ldb2 % 8 == 0 && o.ldb2 >= o.k)),
                 "segment %d: leading dimensions must be multiples of 8 and >= k", s);
    // the kernel addresses a row's 16-byte chunks by 32-bit byte offsets from the plane's start
    auto fits = [](int64_t rows, int64_t ld) { return rows <= 0 || ((rows - 1) * ld + 32) * 2 <= 0xffffffffLL; };
    EG_CHECK_ARG(fits(m, o.lda) && fits(n, o.ldb) && (n2 == 0 || fits(n2, o.ldb2)),
                 "segment %d: a bf16 plane spans 4 GiB or more", s);
    GemmSeg& sg = g.seg[g.n_seg];
    sg.a_hi = (const __bf16*)o.a_hi;
    sg.a_lo = (const __bf16*)o.a_lo;
    sg.b_hi[0] = (const __bf16*)o.b_hi;
    sg.b_lo[0] = (const __bf16*)o.b_lo;
    sg.b_hi[1] = (const __bf16*)(n2 ? o.b2_hi : o.b_hi);
    sg.b_lo[1] = (const __bf16*)(n2 ? o.b2_lo : o.b_lo);
    sg.lda = o.lda;
    sg.ldb[0] = o.ldb;
    sg.ldb[1] = n2 ? o.ldb2 : o.ldb;
    sg.ktiles = o.k / 32;
    ++g.n_seg;
  }
  return EG_OK;
}
}  // namespace
}  // namespace eg

extern "C" {

int eg_gemm_bf16x3(const eg_gemm_operands* ops, int32_t n_seg, int64_t m, int64_t n, int64_t n2, float* c,
                   int64_t ldc, float* c2, int64_t ldc2, int32_t accumulate, int32_t k_slices, void* workspace,
                   int64_t workspace_bytes, void* stream) {
  using namespace eg;
  GemmArgs g{};
  const int rc = bf16_operands(ops, n_seg, m, n, n2, g);
  if (rc != EG_OK) return rc;
  return launch_gemm<kX3BM, kX3BN>(kX3Shape, gemm_x3_kernel<kX3BM, kX3BN, kX3WM, kX3WN, 3>, "gemm_x3_kernel", g, m, n,
                                   n2, c, ldc, c2, ldc2, accumulate, k_slices, workspace, workspace_bytes,
                                   stream);
}

int eg_gemm_bf16x6(const eg_gemm_operands* hi_mid, const eg_gemm_operands* hi_lo, int32_t n_seg, int64_t m,
                   int64_t n, int64_t n2, float* c, int64_t ldc, float* c2, int64_t ldc2, int32_t accumulate,
                   int32_t k_slices, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace eg;
  GemmArgs g1{}, g2{};
  int rc = bf16_operands(hi_mid, n_seg, m, n, n2, g1);
  if (rc != EG_OK) return rc;
  rc = bf16_operands(hi_lo, n_seg, m, n, n2, g2);
  if (rc != EG_OK) return rc;
  bool same = g1.n_seg == g2.n_seg;
  for (int s = 0; same && s < g1.n_seg; ++s) same = g1.seg[s].ktiles == g2.seg[s].ktiles;
  EG_CHECK_ARG(same, "hi_mid and hi_lo must describe the same K segments");
  // One K segment: the six products in one launch, the hi / lo planes as a
  // second segment over the same K (one last round and one sum of its parts;
  // 12 % faster on the PLE key + value), when the workspace covers that
  // launch's plan.  Two K segments keep two launches: one launch's last round
  // of ranges, all of the backward's tiles, mixes steps of four and of two
  // products unevenly (4 % slower).
  if (g1.n_seg == 1) {
    GemmArgs g = g1;
    g.seg[1] = g2.seg[0];
    g.n_seg = 2;
    const int64_t need = workspace_size(kX3Shape, m, n, n2, 2 * 32 * g1.seg[0].ktiles, k_slices);
    if (need >= 0 && workspace_bytes >= need)
      return launch_gemm<kX3BM, kX3BN>(kX3Shape, gemm_x6_kernel<kX3BM, kX3BN, kX3WM, kX3WN>, "gemm_x6_kernel", g, m,
                                       n, n2, c, ldc, c2, ldc2, accumulate, k_slices, workspace, workspace_bytes,
                                       stream);
  }
  // lo*lo + lo*hi + hi*lo + hi*hi over the hi and mid planes, then lo*hi + hi*lo
  // over the hi and lo planes, added to it
  rc = launch_gemm<kX3BM, kX3BN>(kX3Shape, gemm_x3_kernel<kX3BM, kX3BN, kX3WM, kX3WN, 4>, "gemm_x3_kernel<4>", g1,
                                 m, n, n2, c, ldc, c2, ldc2, accumulate, k_slices, workspace, workspace_bytes,
                                 stream);
  if (rc != EG_OK) return rc;
  return launch_gemm<kX3BM, kX3BN>(kX3Shape, gemm_x3_kernel<kX3BM, kX3BN, kX3WM, kX3WN, 2>, "gemm_x3_kernel<2>", g2,
                                   m, n, n2, c, ldc, c2, ldc2, 1, k_slices, workspace, workspace_bytes, stream);
}

}  // extern "C"

namespace eg {
namespace {
// The kernel arguments of eg_gemm_f32(_rows) operands, checked.
int f32_operands(const eg_gemm_f32_operands* ops, int32_t n_seg, int64_t n2, F32Args& g) {
  EG_CHECK_ARG(ops != nullptr && n_seg >= 0 && n_seg <= 2, "n_seg=%d", n_seg);
  for (int s = 0; s < n_seg; ++s) {
    const eg_gemm_f32_operands& o = ops[s];
    EG_CHECK_ARG(o.k >= 0 && o.k % 32 == 0, "segment %d: k must be a multiple of 32 (k=%lld)", s, (long long)o.k);
    if (o.k == 0) continue;
    const float* mats[3] = {o.a, o.b, o.b2};
    for (int q = 0; q < 3; ++q) {
      if (q == 2 && n2 == 0) break;
      EG_CHECK_ARG(mats[q] != nullptr && ((uintptr_t)mats[q] & 15) == 0,
                   "segment %d: operand %d is NULL or not 16-byte aligned", s, q);
    }
    EG_CHECK_ARG(o.lda % 4 == 0 && o.ldb % 4 == 0 && o.lda >= o.k && o.ldb >= o.k &&
                     (n2 == 0 || (o.ldb2 % 4 == 0 && o.ldb2 >= o.k)),
                 "segment %d: leading dimensions must be multiples of 4 and >= k", s);
    F32Seg& sg = g.seg[g.n_seg];
    sg.a = o.a;
    sg.b[0] = o.b;
    sg.b[1] = n2 ? o.b2 : o.b;
    sg.lda = o.lda;
    sg.ldb[0] = o.ldb;
    sg.ldb[1] = n2 ? o.ldb2 : o.ldb;
    sg.ktiles = o.k / 32;
    ++g.n_seg;
  }
  return EG_OK;
}
}  // namespace
}  // namespace eg

extern "C" {

int eg_gemm_f32(const eg_gemm_f32_operands* ops, int32_t n_seg, int64_t m, int64_t n, int64_t n2, float* c,
                int64_t ldc, float* c2, int64_t ldc2, int32_t accumulate, int32_t k_slices, void* workspace,
                int64_t workspace_bytes, void* stream) {
  using namespace eg;
  F32Args g{};
  const int rc = f32_operands(ops, n_seg, n2, g);
  if (rc != EG_OK) return rc;
  return launch_gemm<kF32BM, kF32BN>(kF32Shape, gemm_f32_kernel<kF32BM, kF32BN>, "gemm_f32_kernel", g, m, n, n2,
                                     c, ldc, c2, ldc2, accumulate, k_slices, workspace, workspace_bytes, stream);
}

int eg_gemm_f32_rows(const eg_gemm_f32_operands* ops, int32_t n_seg, int64_t m, int64_t n, int64_t n2, float* c,
                     int64_t ldc, float* c2, int64_t ldc2, int32_t accumulate, void* stream) {
  using namespace eg;
  F32Args g{};
  const int rc = f32_operands(ops, n_seg, n2, g);
  if (rc != EG_OK) return rc;
  EG_CHECK_ARG(m >= 0 && n >= 0 && n2 >= 0, "m=%lld n=%lld n2=%lld", (long long)m, (long long)n, (long long)n2);
  if (m > kFewRows)
    return set_error(EG_ERR_UNSUPPORTED, "eg_gemm_f32_rows of %lld rows (built: up to %d)", (long long)m, kFewRows);
  if (m == 0 || n + n2 == 0) return EG_OK;
  EG_CHECK_ARG(n == 0 || (c != nullptr && ldc >= n), "c / ldc");
  EG_CHECK_ARG(n2 == 0 || (c2 != nullptr && ldc2 >= n2), "c2 / ldc2");
  Plan& p = g.p;
  p.c[0] = c;
  p.c[1] = c2;
  p.ldc[0] = ldc;
  p.ldc[1] = ldc2;
  p.m = m;
  p.n[0] = n;
  p.n[1] = n2;
  p.accumulate = accumulate ? 1 : 0;
  const int64_t blocks = (n + 31) / 32 + (n2 + 31) / 32;
  EG_CHECK_ARG(blocks < (1LL << 31), "too many columns");
  // sixteen wavefronts a workgroup where the columns are fewer than the CUs
  const dim3 grid((unsigned)blocks);
  hipStream_t st = (hipStream_t)stream;
  if (m <= kVecRows) {
    // one group of 4 columns a wavefront fills the 256 CUs with ten or more each from about
    // 10,000 columns on; below, four wavefronts share a group
    const int64_t groups = (n + kVecCols - 1) / kVecCols + (n2 + kVecCols - 1) / kVecCols;
    const bool split = groups < 2560;
    const dim3 vgrid((unsigned)(split ? groups : (groups + 3) / 4));
    auto go = [&](auto rows) {
      constexpr int M = decltype(rows)::value;
      if (split) hipLaunchKernelGGL((gemm_f32_vec_kernel<M, 4>), vgrid, dim3(256), 0, st, g);
      else hipLaunchKernelGGL((gemm_f32_vec_kernel<M, 1>), vgrid, dim3(256), 0, st, g);
    };
    if (m == 1) go(std::integral_constant<int, 1>{});
    else if (m == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
    return launch_status("gemm_f32_vec_kernel");
  }
  if (blocks <= 256 && m <= 8)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<16, 8, 3>), grid, dim3(1024), 0, st, g);
  else if (blocks <= 256)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<16, 32, 2>), grid, dim3(1024), 0, st, g);
  else if (m <= 8)
    hipLaunchKernelGGL((gemm_f32_rows_kernel<8, 8, 3>), grid, dim3(512), 0, st, g);
  else
    hipLaunchKernelGGL((gemm_f32_rows_kernel<8, 32, 2>), grid, dim3(512), 0, st, g);
  return launch_status("gemm_f32_rows_kernel");
}

}  // extern "C"

namespace eg {
namespace {
// One operand of eg_gemm_f16x3, checked: its sources' total of 32-wide K steps.
int f16_matrix(const eg_f16_matrix* x, const char* what, int64_t* steps) {
  EG_CHECK_ARG(x != nullptr && x->rows >= 0 && x->n_src >= 1 && x->n_src <= 2, "%s: rows / n_src", what);
  *steps = 0;
  for (int s = 0; s < x->n_src; ++s) {
    const eg_f16_source& o = x->src[s];
    EG_CHECK_ARG(o.cols >= 0 && o.row_stride >= 0 && o.col_stride >= 0, "%s: source %d", what, s);
    EG_CHECK_ARG(o.x != nullptr || o.cols == 0 || x->rows == 0, "%s: source %d is NULL", what, s);
    *steps += (o.cols + 31) / 32;
  }
  EG_CHECK_ARG(x->rows == 0 || *steps == 0 ||
                   (x->planes != nullptr && ((uintptr_t)x->planes & 15) == 0 && x->exps != nullptr),
               "%s: planes (16-byte aligned) and exps", what);
  return EG_OK;
}

F16Src f16_src(const eg_f16_matrix* x, int s) {
  return s < x->n_src ? F16Src{x->src[s].x, x->src[s].cols, x->src[s].row_stride, x->src[s].col_stride}
                      : F16Src{nullptr, 0, 0, 0};
}

int64_t blocks32(int64_t rows) { return (rows + 31) / 32; }

// exps holds the rows' exponents of source 0, those of source 1, the rows' info of
// either, and the summaries of 8 rows.
int32_t* f16_exps(const eg_f16_matrix* x, int s) { return x->exps + blocks32(x->rows) * 32 * s; }
int32_t* f16_info(const eg_f16_matrix* x, int s) { return x->exps + blocks32(x->rows) * 32 * (2 + s); }
int32_t* f16_sum8(const eg_f16_matrix* x) { return x->exps + blocks32(x->rows) * 128; }
}  // namespace
}  // namespace eg

extern "C" {

int64_t eg_f16_planes_bytes(int64_t rows, int64_t k) { return rows < 0 || k < 0 ? -1 : eg::blocks32(rows) * ((k + 31) / 32) * eg::kStepBytes; }

int64_t eg_f16_exps_count(int64_t rows) { return rows < 0 ? -1 : eg::blocks32(rows) * 140; }

int eg_split_f16(const eg_f16_matrix* x, void* stream) {
  using namespace eg;
  int64_t steps = 0;
  const int rc = f16_matrix(x, "x", &steps);
  if (rc != EG_OK) return rc;
  if (x->rows == 0 || steps == 0) return 0;
  SplitF16Args a{};
  bool trans = false;
  for (int s = 0; s < 2; ++s) {
    a.src[s] = f16_src(x, s);
    a.chunks[s] = (a.src[s].cols + 31) / 32 * 4;
    trans = trans || (a.src[s].cols > 0 && a.src[s].col_stride != 1);
  }
  a.rows = x->rows;
  a.blk = steps * kStepBytes;
  a.planes = (char*)x->planes;
  a.exps[0] = f16_exps(x, 0);
  a.exps[1] = f16_exps(x, 1);
  a.info[0] = f16_info(x, 0);
  a.info[1] = f16_info(x, 1);
  a.sum8 = f16_sum8(x);
  const int64_t blocks = trans ? blocks32(x->rows) : 4 * blocks32(x->rows);
  EG_CHECK_ARG(blocks < (1LL << 31), "too many rows");
  const int64_t chunks = 4 * steps;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)blocks);
  // K kept in registers where it fits a thread's 80 (rows) or 48 (columns;
  // 1,024 threads have 128 registers each, and 64 values spilled) values
  if (trans) {
    if (chunks <= 6 * 16 * 2)
      hipLaunchKernelGGL((split_f16_kernel<32, 16, 6, true>), grid, dim3(1024), 0, st, a);
    else
      hipLaunchKernelGGL((split_f16_kernel<32, 16, 0, true>), grid, dim3(1024), 0, st, a);
  } else {
    if (chunks <= 10 * 4 * 8)
      hipLaunchKernelGGL((split_f16_kernel<8, 4, 10, false>), grid, dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL((split_f16_kernel<8, 4, 0, false>), grid, dim3(256), 0, st, a);
  }
  return launch_status("split_f16_kernel");
}

int eg_gemm_f16x3(const eg_f16_matrix* a, const eg_f16_matrix* b, const eg_f16_matrix* b2, float* c, int64_t ldc,
                  float* c2, int64_t ldc2, void* workspace, int64_t workspace_bytes, void* stream) {
  using namespace eg;
  const eg_f16_matrix none{};
  int64_t ka = 0, kb = 0, kb2 = 0;
  int rc = f16_matrix(a, "a", &ka);
  if (rc == EG_OK) rc = f16_matrix(b, "b", &kb);
  if (rc == EG_OK && b2 != nullptr) rc = f16_matrix(b2, "b2", &kb2);
  if (rc != EG_OK) return rc;
  const eg_f16_matrix* second = b2 != nullptr ? b2 : &none;
  for (int s = 0; s < 2; ++s)
    EG_CHECK_ARG(f16_src(a, s).cols == f16_src(b, s).cols && (b2 == nullptr || f16_src(a, s).cols == f16_src(b2, s).cols),
                 "source %d: a and b must have the same k", s);
  const int64_t m = a->rows, n = b->rows, n2 = second->rows;
  if (m == 0 || n + n2 == 0) return 0;
  H3Args g{};
  if (ka > 0) {
    H3Seg& sg = g.seg[0];
    sg.a = (const char*)a->planes;
    sg.b[0] = (const char*)b->planes;
    sg.b[1] = (const char*)second->planes;
    sg.a_blk = ka * kStepBytes;
    sg.a_blocks = blocks32(m);
    sg.b_blocks[0] = blocks32(n);
    sg.b_blocks[1] = blocks32(n2);
    sg.ktiles = ka;
    g.n_seg = 1;
  }
  const int last = a->n_src - 1;
  g.scale = RowScale{f16_exps(a, last), {f16_exps(b, last), f16_exps(second, last)}};
  g.first = RowScale{f16_exps(a, 0), {f16_exps(b, 0), f16_exps(second, 0)}};
  g.kt_first = last > 0 ? (a->src[0].cols + 31) / 32 : ka;
  EG_CHECK_ARG(ka > 0, "k must be positive");
  const bool two = g.kt_first > 0 && g.kt_first < ka;
  rc = launch_gemm<kX3BM, kX3BN>(two ? kH3TwoShape : kX3Shape,
                                 two ? gemm_h3_kernel<kX3BM, kX3BN, kX3WM, kX3WN, true>
                                     : gemm_h3_kernel<kX3BM, kX3BN, kX3WM, kX3WN, false>,
                                 "gemm_h3_kernel", g, m, n, n2, c, ldc, c2, ldc2, 0, 0, workspace, workspace_bytes,
                                 stream, g.scale);
  if (rc != EG_OK) return rc;
  WideArgs w{};
  for (int s = 0; s < 2; ++s) {
    w.a[s] = f16_src(a, s);
    w.b[0][s] = f16_src(b, s);
    w.b[1][s] = f16_src(second, s);
  }
  w.n_src = a->n_src;
  const eg_f16_matrix* of[3] = {a, b, second};
  for (int x = 0; x < (b2 != nullptr ? 3 : 2); ++x) {
    w.info[x][0] = f16_info(of[x], 0);
    w.info[x][1] = f16_info(of[x], 1);
    w.sum8[x] = f16_sum8(of[x]);
  }
  for (int s = 0; s < 2; ++s) {
    const int64_t k = w.a[s].cols;
    w.near[s] = (int)std::min<int64_t>(k + (k + kNearShare - 1) / kNearShare, INT32_MAX);
  }
  w.m = m;
  w.n[0] = n;
  w.n[1] = n2;
  w.c[0] = c;
  w.c[1] = c2;
  w.ldc[0] = ldc;
  w.ldc[1] = ldc2;
  hipLaunchKernelGGL(gemm_wide_kernel, dim3(kWideGroups), dim3(64 * kWideWaves), 0, (hipStream_t)stream, w);
  return launch_status("gemm_wide_kernel");
}

}  // extern "C"
