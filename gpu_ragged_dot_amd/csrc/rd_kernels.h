// Grouped-GEMM kernels built on gemm_tile(): launch-index -> tile mapping, group lookup through the scheduling
// map, tail / empty-group zeroing.
#pragma once
#include "rd_gemm_dlds.h"
#include "rd_gemm_f32.h"
#include "rd_gemm_f8.h"
#include "rd_gemm_w4.h"
#include "rd_gemm_w4r.h"
#include "rd_gemm_ws.h"
#include "rd_gemm_pp.h"
#include "rd_gemm_rs.h"
#include "rd_gemm_tile.h"
#include "rd_lookup.h"
#include "rd_sched.h"

namespace rd {

// y[m, n] = ragged x[m, k] . A[g]  (A is [g, k, n], or [g, n, k] when trans_rhs).
struct GmmArgs {
  const void* x;  // element type is the kernel configuration's Elem (bf16 bits or float)
  const void* A;
  void* y;
  const int32_t* group_sizes;    // [g]
  const int32_t* group_offsets;  // [g]   exclusive prefix sum of group_sizes
  const int32_t* tile2group;     // [U]   scheduling map built with chunk = tile height
  const int32_t* tile2it;        // [U]
  const int32_t* tile2band;      // [U]   band of row tiles each row tile belongs to (see rd_sched.h)
  const int32_t* total_tiles;    // [1]   null: no map was built, every work-group looks its tile up itself (rd_lookup.h)
  int m, k, n, g;  // g: all groups of group_sizes
  int g_first, g_local;  // A holds the g_local groups [g_first, g_first + g_local); rows of the others are zero
  int U;        // static bound on row tiles: ceil(m / BM) + g
  int n_tiles;  // ceil(n / BN)
  int group_m, group_n;  // tile walk: most row tiles per band; positions per block = group_m x group_n
  // K-split of the last, partly filled round of tiles (kernels whose configuration has SPLITK; 0 slots = off)
  float* partials;     // [split_slots][BM * BN] fp32
  int32_t* counters;   // [split_slots], zero at launch
  int split_slots;     // work-groups appended to the launch for the split pieces
  int max_parts;       // > 0: most pieces a tile is cut into, as the caller asked; 0: chosen from k
  int num_cus;         // tiles the device runs at a time (one work-group per compute unit)
  int main_grid;       // launch indices below this walk whole tiles (set by the launcher)
  // order in which the blocks of the walk are dealt (see launch_sched_map; null: walk order)
  const int32_t* block_order;
  int n_blocks;
};

// dA[g, k, n] = x[rows of g, k]^T . dy[rows of g, n]
struct TgmmArgs {
  const void* x;
  const void* dy;
  void* dA;
  const int32_t* group_sizes;
  const int32_t* group_offsets;  // null: every work-group adds up the sizes before its group itself
  int m, k, n, g;  // g: groups of dA (the slices computed)
  int g_first;     // dA[i] belongs to group g_first + i of group_sizes / group_offsets
  int k_tiles, n_tiles;  // ceil(k / BM), ceil(n / BN)
  int group_m;
  bool edge_lines;  // the launch takes the kernel that stores the lines at its tiles' edges apart, where it has one (kEdgeLineRows)
  const int32_t* group_order;  // null, or the records of the order in which the launch visits the groups (launch_sched_map)
};

// A value every lane holds identically, moved to a scalar register.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <class C, class = void>
struct IsW4 { static constexpr bool value = false; };
template <class C>
struct IsW4<C, decltype((void)C::W4)> { static constexpr bool value = true; };
template <class C, class = void>
struct IsW4R { static constexpr bool value = false; };
template <class C>
struct IsW4R<C, decltype((void)C::W4R)> { static constexpr bool value = true; };

template <class C, class = void>
struct IsMixed { static constexpr bool value = false; };
template <class C>
struct IsMixed<C, typename std::enable_if<C::MIXED>::type> { static constexpr bool value = true; };

// Element type of a configuration's output: its Out when it names one (float8 operands give bf16), else that of its operands.
template <class C, class = void>
struct OutOf { typedef typename C::Elem type; };
template <class C>
struct OutOf<C, decltype((void)sizeof(typename C::Out))> { typedef typename C::Out type; };

constexpr int kW4RMinK = 1792;  // measured: level at 1536, 7 % ahead at 2048, 13 % at 8192 (eight groups of 2048 rows)

template <class C, bool EDGE_LINES = false>
__device__ __forceinline__ void run_tile(const typename C::Elem* Ap, int lda, int a_lim, const typename C::Elem* Bp,
                                         int ldb, int b_lim, int klen, typename OutOf<C>::type* Op, int ldo,
                                         typename C::Elem* smem, const SplitK& sk = SplitK()) {
  if constexpr (C::F32) gemm_tile_f32<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem);
  else if constexpr (IsRs<C>::value) gemm_tile_rs<C, EDGE_LINES>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, reinterpret_cast<unsigned char*>(smem), sk);
  else if constexpr (IsF8Direct<C>::value) {
    if constexpr (C::PINGPONG) gemm_tile_f8_pingpong<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
    else gemm_tile_f8<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  }
  else if constexpr (IsW4R<C>::value) {
    // The register-staged form has four 64-wide slabs to fill before it runs and pays for that on a short contraction:
    // below kW4RMinK the 32-wide direct-to-LDS form of the same core takes the tile.
    if (klen >= kW4RMinK) gemm_tile_w4r<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
    else gemm_tile_w4<W4Cfg<C::BM, C::BN, true, true, 5, C::HALF>>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  }
  else if constexpr (IsWs<C>::value) gemm_tile_ws<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  else if constexpr (IsW4<C>::value) gemm_tile_w4<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  else if constexpr (C::MIXED) gemm_tile_pingpong_mixed<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  else if constexpr (C::DLDS && C::PINGPONG) gemm_tile_pingpong<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  else if constexpr (C::DLDS) gemm_tile_dlds<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, smem, sk);
  else gemm_tile<C>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, Op, ldo, reinterpret_cast<bf16_bits*>(smem));
}

// Row tiles of a group with at most kShortRows rows (most tiles of a launch when the groups are much shorter than the
// tile: a mixture of experts with a few dozen tokens per expert).  Such a tile is a stream over its 256 columns of the
// group's weights with next to no matrix-core work, so what counts is how many bytes each compute unit keeps in flight
// and that every load covers whole 128-byte lines: the same 256 threads run a 64-row tile routine instead, whose LDS
// ring holds only 4-8 KB of activations per slab - 8 slabs of 32 deep for weights read across rows (7 x 20 KB requested
// ahead of use against 3.5 x 32 KB in the tall routine), 4 slabs of 64 deep for weights read along rows.  The weights
// of such a group are read by this one row tile only: they are streamed past L2 (nt), which keeps L2 for what the
// tall tiles of long groups share.
// A 128-row routine of the same kind (6 slabs of 32, or 3 of 64) serves the tiles with 65 to 128 rows.
constexpr int kShortRows = 64, kMidRows = 128;
template <class C, int ROWS>
struct ShortTileCfg {
  static constexpr int BK = C::B_KMAJOR ? 64 : 32;
  static constexpr int STAGES = (160 * 1024) / ((ROWS + C::BN) * BK * 2);
  typedef DldsCfg<ROWS, C::BN, BK, 1, 4, true, C::B_KMAJOR, STAGES, false, kCachePolicyStream, C::HALF> type;
};

// What a cut is worth depends on the core: its K loop per contraction index and how much a piece's partial sums are.
// QUARTERS: the former over the latter, in quarters of the 256 x 256 bf16 cores' (float8: twice the rate; float32
// as three bf16 terms: 6 times the time per multiplication, partial sums of half a tile or a quarter; on the float32 instruction 16 times).
// MIN_K: contraction indices a piece must keep.  float32 rounded to bf16 stays at the bf16 cores' limit (cut from k = 3700 on, 8192 x
// 4096 x 4096 in 8 groups went from 377 to 429 us: its 256 x 256 pieces cost what a bf16 core's do).
template <class C, class = void>
struct SplitCost { static constexpr int QUARTERS = sizeof(typename C::Elem) == 1 ? 2 : 4, MIN_K = 512; };
// The tiles of rd_gemm_ws.h have a sixteenth to half the partial sums: cut from k = 3658 on where few tiles are expected, from 5700
// on always (kWsCutMinK in rd_capi.hip); three pieces already bring most of it.  492 x 4848 x 272 in 19 groups 35 -> 23 us, 720 x
// 4016 x 352 in 9 31 -> 21, 259 x 10432 x 336 in 3 56 -> 21; 477 x 5920 x 3120 in 4 (128 x 128) 54 -> 40.
template <class C>
struct SplitCost<C, typename std::enable_if<IsWs<C>::value>::type> { static constexpr int QUARTERS = 7, MIN_K = 1280; };
template <class C>
struct SplitCost<C, typename std::enable_if<IsRs<C>::value>::type> {
  static constexpr int QUARTERS = C::FULL ? 32 : C::THREE ? 24 : 4, MIN_K = C::FULL || C::THREE ? 256 : 512;
};

// Whether a launch computes the tiles of its last, partly filled round in halves of the columns, on the same core's tile of half the width.
template <class C, class = void>
struct HalvesLastRound { static constexpr bool value = false; };
template <class C>
struct HalvesLastRound<C, typename std::enable_if<IsRs<C>::value>::type> { static constexpr bool value = C::THREE && C::BN == 256 && C::A_KMAJOR; };

// Which launches are cut by split_parts_by_gain(); the others by the square root of the K loop over what a piece costs.
template <class C>
struct SplitsByGain { static constexpr bool value = C::SPLITK && C::DLDS && C::BM * C::BN == 256 * 256; };

// Walk tiles in bands of `group_m` rows: consecutive ids share B columns / A rows so that the ~32 tiles one XCD
// has in flight re-use each other's operands out of its L2.
__device__ __forceinline__ void band_walk(int id, int rows, int cols, int group_m, int& ri, int& cj) {
  const int band_sz = group_m * cols;
  const int band = id / band_sz;
  const int within = id - band * band_sz;
  const int gm = imin(group_m, rows - band * group_m);
  cj = within / gm;
  ri = band * group_m + (within - cj * gm);
}

// trans_rhs: the tiles that stream their weights begin at different slabs (gemm_tile_dlds()) where the weights' row pitch in
// elements is a multiple of this.  us, all from slab 0 | spread: 2048 rows in 128 groups of 16: k 2048, n 768 93 | 73, n 1024 121 |
// 89, n 7168 675 | 584, k 4096, n 768 172 | 137; 1024 rows in 64, n 1024: k 6144 152 | 126.  At other pitches, same rows: k 1536,
// 1792, 2176, 2304, 2560, 5120, 7168 level, 3584 76 | 77, 3072 67 | 74.
constexpr int kRotatePitch = 2048;

template <class C, bool TRANS_RHS>
__global__ __launch_bounds__(C::NT, C::WAVES_PER_EU) void gmm_kernel(GmmArgs p) {
  typedef typename C::Elem E;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  E* smem = reinterpret_cast<E*>(smem_raw);
  const E* px = static_cast<const E*>(p.x);
  const E* pA = static_cast<const E*>(p.A);
  typedef typename OutOf<C>::type O;
  O* py = static_cast<O*>(p.y);
  // Tile walk.  The scheduling-map kernel has cut every group's row tiles into bands of at most group_m row tiles
  // (tile2band); the walk visits band after band and, inside a band, column after column (all the band's row tiles of
  // one column tile, then the next column).  Position t of the walk therefore lies in the band of row tile t / n_tiles.
  // The walk is cut into blocks of group_m x group_n consecutive positions - a band's rows times a few columns, about
  // what one XCD runs at a time, so the block's operand slabs are fetched into that XCD's L2 once - and the blocks are
  // dealt to the 8 XCDs (launch index mod 8) round-robin.  No block spans two groups' weights except where a band ends.
  // Everything read through the map is the same for the whole work-group: pin it to scalar registers.
  const bool mapped = p.total_tiles != nullptr;
  GroupScan<C::BM> scan;
  if (!mapped) scan.init(p.group_sizes, p.g);
  const int total = imin(mapped ? uniform(*p.total_tiles) : scan.total_tiles, p.U);
  const int live = total * p.n_tiles;
  SplitPlan sp{live, 1, 0};
  if constexpr (C::SPLITK) {
    const SplitRule rule{p.k, (int)((long long)p.k * SplitCost<C>::QUARTERS / 4), SplitCost<C>::MIN_K, p.split_slots, p.num_cus, p.max_parts, SplitsByGain<C>::value};
    sp = split_plan(live, rule, HalvesLastRound<C>::value ? 2 : 1);
  }

  int t, half = 0;
  SplitK sk;
  int k0 = 0, klen = p.k;
  if ((int)blockIdx.x < p.main_grid) {
    // With only a few rounds of tiles, blocks of the full size would leave some XCDs without work (180 tiles in blocks
    // of 32 occupy 6 of the 8): the blocks shrink so that every round deals one to each XCD.
    int per_block = p.group_m * p.group_n;
    bool whole_blocks = true;
    if (live < 4 * p.num_cus) {
      const int rounds = (live + p.num_cus - 1) / p.num_cus;
      const int fewer = imax(1, imin(per_block, (live + 8 * rounds - 1) / (8 * rounds)));
      whole_blocks = fewer == per_block;
      per_block = fewer;
    }
    const int pos = blockIdx.x >> 3;
    int block = (pos / per_block) * 8 + (blockIdx.x & 7);
    // Groups much longer than a tile (matrix-core-bound tiles) and groups shorter than one (tiles that stream their
    // group's weights) in one launch: their blocks are dealt interleaved instead of in the order the groups come in, so
    // that at any time some of every XCD's compute units multiply while the others stream (DeepSeek-V3 shape, dlhs:
    // 1.63 -> 1.55 ms; all long groups first, or all short ones, is slower than either).  Same tiles, same results.
    if (p.block_order && whole_blocks) {
      const int n_long = uniform(p.block_order[0]), n_live = uniform(p.block_order[1]);
      bool from_long;
      int rank;
      if (interleaved_slot(block, n_long, n_live, &from_long, &rank))
        block = uniform(p.block_order[from_long ? 2 + rank : 2 + p.n_blocks - 1 - rank]);
    }
    t = block * per_block + pos % per_block;
    if (t >= p.U * p.n_tiles) return;
    if (t >= sp.first_tile && t < live) return;  // computed in pieces by the appended work-groups
  } else {
    // Piece `part` of split tile tt.  The pieces are numbered part-major (all tiles of the first K range, then the
    // second ...) and every XCD (launch index mod 8) takes one contiguous stretch of that numbering, so that the pieces
    // an XCD runs together are neighbouring tiles of one K range and share their operand slabs in its L2.
    const int r = blockIdx.x - p.main_grid;
    const int pieces = sp.tiles * sp.parts;
    const int per_xcd = (pieces + 7) >> 3;
    if ((r >> 3) >= per_xcd) return;
    const int id = (r & 7) * per_xcd + (r >> 3);
    if (id >= pieces) return;
    const int part = id / sp.tiles, tt = id - part * sp.tiles;
    t = sp.first_tile + tt;
    if constexpr (HalvesLastRound<C>::value) { t = sp.first_tile + (tt >> 1); half = tt & 1; }
    const int k64 = (p.k + 63) >> 6;
    k0 = (int)((long long)k64 * part / sp.parts) << 6;
    klen = imin(p.k, (int)((long long)k64 * (part + 1) / sp.parts) << 6) - k0;
    sk.partials = p.partials + (size_t)tt * sp.parts * (C::BM * C::BN / (HalvesLastRound<C>::value ? 2 : 1));
    sk.counter = p.counters + tt;
    sk.parts = sp.parts;
    sk.part = part;
  }
  const int walk_row = t / p.n_tiles;
  bool deferred = false;  // a short last row tile the map has moved behind all other tiles
  int band_row0 = walk_row, band_rows = 1;
  int gi = 0, first_row = 0, group_rows = 0, first_tile = 0;  // of the tile's group, where there is no map
  if (mapped) {
    const int band = uniform(p.tile2band[walk_row]);
    deferred = (band & kBandDeferred) != 0;
    band_row0 = (band & ~kBandDeferred) >> kBandShift;
    band_rows = band & kBandMaxRows;
  } else if (walk_row < total) {
    scan.find(walk_row, &gi, &group_rows, &first_row, &first_tile);
    int first;
    band_of((group_rows + C::BM - 1) / C::BM, p.group_m, walk_row - first_tile, &first, &band_rows);
    band_row0 = first_tile + first;
  }
  const int w = t - band_row0 * p.n_tiles;
  const int nj = w / band_rows;
  const int mi = band_row0 + (w - nj * band_rows);
  const int col0 = nj * C::BN + half * (C::BN / 2);
  const int cols = imin(HalvesLastRound<C>::value && t >= sp.first_tile && t < live ? C::BN / 2 : C::BN, p.n - col0);
  if (cols <= 0) return;  // the second half of a tile of few columns

  if (mi < total) {
    int it = mi - first_tile;
    if (mapped) {
      gi = uniform(p.tile2group[mi]);
      it = uniform(p.tile2it[mi]);
      first_row = uniform(p.group_offsets[gi]);
      group_rows = uniform(p.group_sizes[gi]);
    }
    const int row0 = first_row + it * C::BM;
    int rows = imin(C::BM, group_rows - it * C::BM);
    rows = imin(rows, p.m - row0);  // group_sizes summing past m: never touch rows >= m
    if (rows <= 0 || row0 < 0) return;
    O* Op = py + (size_t)row0 * p.n + col0;
    const int gl = gi - p.g_first;  // index of the group's weights in A
    if (gl < 0 || gl >= p.g_local) {
      // a group whose weights live elsewhere (A is a slice of the groups): its rows of y are zero
      if (sk.part == 0) zero_tile<C::NT, C::VEC, O>(Op, p.n, rows, cols);
      return;
    }
    const E* Ap = px + (size_t)row0 * p.k + k0;
    const E* Bp = TRANS_RHS ? pA + (size_t)gl * p.n * p.k + (size_t)col0 * p.k + k0
                            : pA + (size_t)gl * p.k * p.n + (size_t)k0 * p.n + col0;
    if constexpr (IsW4<C>::value && C::A_KMAJOR) {
      // For a group's single row tile, and for the short last tile of a longer group where the scheduling map has moved
      // it behind all other tiles (into the K-split last round).  Left in its group's run such a tile must stay on the tall routine: run
      // through the short one it finishes early, the tiles dealt next start out of step with the rest of their block,
      // and the block's operand slabs are fetched into L2 twice (measured: +1 GB of fetches per launch, no time gained).
      if (rows <= kMidRows && (it == 0 || deferred)) {
        typedef typename ShortTileCfg<C, kShortRows>::type S;
        typedef typename ShortTileCfg<C, kMidRows>::type M;
        static_assert(S::LDS_BYTES <= C::LDS_BYTES && S::NT == C::NT && S::BN == C::BN, "the short routine runs in the tall one's launch");
        static_assert(M::LDS_BYTES <= C::LDS_BYTES && M::NT == C::NT && M::BN == C::BN, "the 128-row routine runs in the tall one's launch");
        const int ldb = TRANS_RHS ? p.k : p.n;
        // from the group, not the tile's place in the launch: a row's sums are added up in an order that the other groups'
        // sizes do not change (odd factor: neighbouring tiles start far apart)
        const uint32_t start = p.k % kRotatePitch == 0 ? (uint32_t)(gi * p.n_tiles + nj) * 13u : 0u;
        if (rows <= kShortRows) gemm_tile_dlds<S>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk, start);
        else gemm_tile_dlds<M>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk, start);
        return;
      }
    }
    if constexpr (IsWs<C>::value) {
      if constexpr (C::STREAMS) {
        // a group's only row tile: nothing else reads its weights (streams_weights() in rd_capi.hip says when).  A kernel of
        // its own: the loops of the tile of 128 x 256 fill the register file, and launches that do not stream stay as they are
        if (it == 0 && group_rows <= C::BM) {
          gemm_tile_ws<C, kCachePolicyStream>(Ap, p.k, rows, Bp, TRANS_RHS ? p.k : p.n, cols, klen, Op, p.n, smem, sk);
          return;
        }
      }
    }
    if constexpr (IsMixed<C>::value) {
      // The eight-wave core with a ring per operand: every row tile of at most 128 rows, a group's only one or its last, on
      // eight-wave routines of 64 or 128 rows with 64-wide slabs of both operands, four or three of them in LDS.  On the tall
      // routine such a tile takes about as long as a whole one: its waves skip their matrix-core work, but the launch pays the
      // slab for slab hand-over of 256 rows.  Unlike on the four-wave core it pays for last tiles too: these routines keep the
      // weights in L2 for the neighbouring tiles (no streaming policy).  Over 75 calls (4282 - 32768 rows, k and n of 448 - 8064, 4
      // - 131 groups) 0.987 (gmm) and 0.983 times (trans_rhs) what the core took without them; with the 64-row routine
      // alone 0.992 and 0.989, with the tall core's own schedule on 128 rows 0.991 and 0.986.  us, before | now: 11122 x 1088 x
      // 768 in 64 skewed groups 52 | 46, trans_rhs 56 | 49; trans_rhs 26452 x 704 x 3712 in 46 199 | 177; 23628 x 2528 x
      // 2112 in 218 skewed groups 548 | 505.
      typedef DldsCfg<kShortRows, C::BN, 64, 2, 4, true, C::B_KMAJOR, 4, false, 0, C::HALF> S;
      typedef DldsCfg<kMidRows, C::BN, 64, 2, 4, true, C::B_KMAJOR, 3, false, 0, C::HALF> M;
      static_assert(S::LDS_BYTES <= C::LDS_BYTES && S::NT == C::NT, "the short routine runs in the tall one's launch");
      static_assert(M::LDS_BYTES <= C::LDS_BYTES && M::NT == C::NT, "the 128-row routine runs in the tall one's launch");
      if (rows <= kMidRows) {
        const int ldb = TRANS_RHS ? p.k : p.n;
        if (rows <= kShortRows) gemm_tile_dlds<S>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk);
        else gemm_tile_dlds<M>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk);
        return;
      }
    }
    if constexpr (IsF8Direct<C>::value) {
      if constexpr (C::NW == 8 && C::WAVES_M == 2 && C::A_KMAJOR && C::BM > kShortRows) {
        // a group's single row tile of at most kShortRows rows, as above: a 64-row routine on 128-deep slabs (every load
        // covers whole 128-byte lines), the weights streamed past L2 - where the tall routine's LDS has room for its ring
        typedef F8Cfg<kShortRows, C::BN, 2, 4, 3, 128, kCachePolicyStream, true, C::B_KMAJOR, false> S;
        if constexpr (S::LDS_BYTES <= C::LDS_BYTES) {
          static_assert(S::NT == C::NT, "the short routine runs in the tall one's launch");
          if (rows <= kShortRows && it == 0) {
            gemm_tile_f8<S>(Ap, p.k, rows, Bp, TRANS_RHS ? p.k : p.n, cols, klen, Op, p.n, smem, sk);
            return;
          }
        }
      }
    }
    if constexpr (HalvesLastRound<C>::value) {
      if (t >= sp.first_tile) {
        typedef RsCfg<C::BM, C::BN / 2, true, C::B_KMAJOR, E, C::VEC, C::FULL, C::THREE, C::WAVES_N> H;
        static_assert(H::LDS_BYTES <= C::LDS_BYTES && H::NT == C::NT, "runs in the whole tile's launch");
        const int ldb = TRANS_RHS ? p.k : p.n;
        if (!rs_short_tile<H>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk)) run_tile<H>(Ap, p.k, rows, Bp, ldb, cols, klen, Op, p.n, smem, sk);
        return;
      }
    }
    if constexpr (IsRs<C>::value) {
      // A group's only row tile, and a few rows behind whole ones (8192 x 4096 x 4096 in 8 groups of about 1024 rows, float32
      // in bf16, half of them a few rows over: 403 -> 387 us, 417 -> 398 with trans_rhs).  Taller last tiles stay on the
      // whole routine: out of step with their neighbours they cost more in shared operand slabs than they save (4096 x
      // 4096 x 4096 in 16: 323 us, 337 with every height cut).
      if ((it == 0 || rows <= 64) && rs_short_tile<C>(Ap, p.k, rows, Bp, TRANS_RHS ? p.k : p.n, cols, klen, Op, p.n, smem, sk)) return;
    }
    run_tile<C>(Ap, p.k, rows, Bp, TRANS_RHS ? p.k : p.n, cols, klen, Op, p.n, smem, sk);
  } else {
    // Rows past sum(group_sizes) are defined to be zero.  The map never uses more than
    // U - ceil(tail / BM) entries, so the unused tile slots cover the tail.
    long long s = mapped ? (long long)uniform(p.group_offsets[p.g - 1]) + uniform(p.group_sizes[p.g - 1]) : scan.total_rows;
    if (s < 0) s = 0;
    const long long r0 = s + (long long)(mi - total) * C::BM;
    if (r0 >= p.m) return;
    const int rows = imin(C::BM, p.m - (int)r0);
    zero_tile<C::NT, C::VEC, O>(py + (size_t)r0 * p.n + col0, p.n, rows, cols);
  }
}

// tgmm tiles of at most this many rows (16-bit results) store the lines at their edges plainly where the rows of dA are no whole number of
// 64-byte halves of a line (store_accumulators()) and the groups average no more (tgmm_impl()).  A kernel of its own: in one
// kernel for both the mere branch cost launches with whole lines 1 to 3 %, those of the four-wave 256 x 256 core 5 %.  Times with over
// without, geometric means over 1640 random calls with such rows, groups averaging under 20 | 20 to 40 | 40 to 60 | 60 to 80 | 80 to
// 120 | 120 to 400 rows:
//   128 x 128, three work-groups to a unit    0.66 | 0.70 | 0.81 | 0.81 | 0.90 | 0.97
//   128 x 256 of rd_gemm_ws.h, bf16           0.78 | 0.85 | 0.86 | 0.93 | 0.97 | 1.00
//                              float16        0.78 | 0.79 | 0.88 | 0.92 | 0.95 | 1.00
//   128 x 128 of rd_gemm_ws.h                 0.81 | 0.87 | 0.93 | 0.93 | 0.99 | 1.00
//   256 x 256, float8                         0.87 | 0.89 | 0.90 | 0.92 | 0.99 | 1.03
// 364 x 5376 x 9584 in 33 groups (128 x 128) 1412 -> 955 us, 2640 x 2048 x 1000 in 33 60 -> 39.  Rows of whole halves: 1.04, up to 1.3
// (7459 x 14112 x 544 in 199 groups 933 | 996).  Not for the bf16 and float16 256 x 256 cores, whose tiles are for longer groups.
//
// float32 results of the any-pitch core: a half wave stores 32 columns of a row at a time, so that inside a tile too every line goes out in two
// parts where rows are no whole number of halves.  Those tiles are stored plainly altogether.  Times with over without, 1100 to 1700 random
// calls with such rows, by rows of a group 4 to 20 | 20 to 40 | 40 to 60 | 60 to 80 | 80 to 100 | 100 to 120 | 120 to 160 | 240 to 400:
//   rounded to bf16, 128 x 128, multiples of 8    0.70 | 0.69 | 0.73 | 0.79 | 0.82 | 0.84 | 0.89 | 0.95
//                    256 x 256                    0.64 | 0.61 | 0.65 | 0.69 | 0.72 | 0.73 | 0.76 | 0.84
//                    128 x 128, other pitches     0.61 | 0.63 | 0.62 | 0.69 | 0.74 | 0.73 | 0.76 | 0.89
//                    256 x 256                    0.57 | 0.57 | 0.56 | 0.61 | 0.68 | 0.62 | 0.66 | 0.80
//   as terms, 128 x 256                           0.76 | 0.84 | 0.84 | 0.89 | 0.93 | 0.92 | 0.95 | 0.99
//   as terms, 128 x 128                           0.98 | 1.05 | 1.04 | 1.05 | 1.04 | 1.03 | 1.02 | 1.01   (not for this one, nor for
//   float32 instruction, 64 x 64                  1.03 | 1.05 | 1.05 | 1.05 | 1.04 | 1.02 | 1.01 | 0.99    this one)
// Rounded to bf16, us: 50 x 5112 x 13016 in 6 groups 779 -> 345 (64 x 64 tile 392), 606 x 3928 x 2472 in 72 1253 -> 662 (717), 270 x 1050 x 14931
// in 3 139 -> 64 (83).
constexpr int kEdgeLineRows = 80, kEdgeLineRowsF32 = 120;
template <class C, class = void>
struct StoresEdgeLines { static constexpr bool value = IsF8Direct<C>::value || IsWs<C>::value; };
template <class C>
struct StoresEdgeLines<C, typename std::enable_if<C::DLDS && !C::PINGPONG && !IsF8Direct<C>::value && !IsWs<C>::value>::type> {
  static constexpr bool value = !IsW4<C>::value && !IsW4R<C>::value;
};
template <class C>
struct StoresEdgeLines<C, typename std::enable_if<IsRs<C>::value>::type> {
  static constexpr bool value = sizeof(typename C::Elem) == 4 && !C::FULL && !(C::THREE && C::BN < 256);
};

template <class C, bool EDGE_LINES = false>
__global__ __launch_bounds__(C::NT, C::WAVES_PER_EU) void tgmm_kernel(TgmmArgs p) {
  typedef typename C::Elem E;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  E* smem = reinterpret_cast<E*>(smem_raw);
  // Work per tile is proportional to its group's row count, which only the device knows and which can be wildly
  // skewed.  So every XCD (launch index mod 8) takes one eighth of every group's tiles - a contiguous stretch of the
  // group's banded walk, so its tiles still share operand columns in its L2 - and all XCDs get the same share of every
  // group however the rows are distributed.
  const int per_group = p.k_tiles * p.n_tiles;
  const int quota = (per_group + 7) >> 3;  // tiles of one group per XCD
  const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3;
  const int slot = pos / quota;
  if (slot >= p.g) return;
  // groups are visited by falling size class, so that tiles of about equal duration run side by side; the record of
  // a position holds the group, its first row and its row count
  int gi = slot, row0, rows;
  if (p.group_order) {
    const int32_t* rec = p.group_order + 4 * (size_t)slot;
    gi = uniform(rec[0]); row0 = uniform(rec[1]); rows = uniform(rec[2]);
  } else {
    row0 = p.group_offsets ? uniform(p.group_offsets[slot + p.g_first]) : rows_before_group(p.group_sizes, slot + p.g_first);
    rows = uniform(p.group_sizes[slot + p.g_first]);
  }
  const int t = ((xcd + slot) & 7) * quota + (pos - slot * quota);
  if (gi < 0 || gi >= p.g || t >= per_group) return;
  int ri, cj;
  band_walk(t, p.k_tiles, p.n_tiles, p.group_m, ri, cj);

  const int kk0 = ri * C::BM, col0 = cj * C::BN;
  const int krows = imin(C::BM, p.k - kk0), cols = imin(C::BN, p.n - col0);
  typedef typename OutOf<C>::type O;
  O* Op = static_cast<O*>(p.dA) + (size_t)gi * p.k * p.n + (size_t)kk0 * p.n + col0;

  rows = imin(rows, p.m - row0);
  if (rows <= 0 || row0 < 0) {  // empty group: its slice of dA is zero
    zero_tile<C::NT, C::VEC, O>(Op, p.n, krows, cols);
    return;
  }
  const E* Ap = static_cast<const E*>(p.x) + (size_t)row0 * p.k + kk0;
  const E* Bp = static_cast<const E*>(p.dy) + (size_t)row0 * p.n + col0;
  SplitK sk;
  sk.edge_lines = EDGE_LINES && rows <= (sizeof(O) == 4 ? kEdgeLineRowsF32 : kEdgeLineRows);
  run_tile<C, EDGE_LINES>(Ap, p.k, krows, Bp, p.n, cols, rows, Op, p.n, smem, sk);
}

// ---- host-side launchers, one set per compiled tile shape -------------------------------------------------------

typedef int (*gmm_launch_fn)(hipStream_t, const GmmArgs&);
typedef int (*tgmm_launch_fn)(hipStream_t, const TgmmArgs&);

struct TileVariant {
  const char* name;
  int bm, bn, bk, waves_m, waves_n;
  int vec;  // 1: needs k % 8 == 0 and n % 8 == 0 (16-byte row pitches); 0: any shape
  int dtype;   // RD_DTYPE_* of the operands and the output this shape is compiled for
  int dlds;    // 1: direct-to-LDS core (byte extents of one tile's operand window must stay below 2 GiB)
  int stages;  // LDS ring depth
  int any_pitch_core;  // 1: the register-staged core of rd_gemm_rs.h (k >= 8, n >= 8, 32-bit offsets within 256 rows)
  int splitk;  // 1: the gmm kernels can cut the last round of tiles along K (needs partials in the workspace)
  int split_quarters, split_min_k;  // SplitCost of the gmm kernels
  int split_bn;  // columns of a piece of the K-split
  int split_by_gain;  // SplitsByGain of the gmm kernels
  int ws_core;  // 1: the core of rd_gemm_ws.h
  int split_rings;  // 1: the core of rd_gemm_pp.h with a ring per operand
  gmm_launch_fn gmm_nn, gmm_nt;  // null: the shape has no kernel for that product
  tgmm_launch_fn tgmm;
  gmm_launch_fn gmm_nn_stream, gmm_nt_stream;  // the same products, the weights of groups of one row tile streamed past the caches; null: no such kernel
};

// Kernels that use more than 64 KB of LDS must opt in, once per device.
static inline int allow_big_lds(const void* kern, int bytes) {
  if (bytes <= 64 * 1024) return hipSuccess;
  return (int)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <class C, bool TRANS_RHS>
int launch_gmm(hipStream_t s, const GmmArgs& a) {
  auto kern = gmm_kernel<C, TRANS_RHS>;
  const int attr_rc = allow_big_lds(reinterpret_cast<const void*>(kern), C::LDS_BYTES);
  if (attr_rc != hipSuccess) return attr_rc;
  // positions per XCD: enough for any block size the kernel may shrink to (at most group_m x group_n)
  const int per_block = a.group_m * a.group_n;
  GmmArgs args = a;
  args.main_grid = 8 * ((a.U * a.n_tiles + 7) / 8 + 2 * per_block);
  if (!C::SPLITK) args.split_slots = 0;
  const int grid = args.main_grid + args.split_slots;
  if (args.main_grid <= 0) return hipSuccess;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::NT), C::LDS_BYTES, s, args);
  return (int)hipGetLastError();
}

template <class C>
int launch_tgmm(hipStream_t s, const TgmmArgs& a) {
  auto kern = tgmm_kernel<C>;
  if constexpr (StoresEdgeLines<C>::value)
    if (a.edge_lines) kern = tgmm_kernel<C, true>;
  const int attr_rc = allow_big_lds(reinterpret_cast<const void*>(kern), C::LDS_BYTES);
  if (attr_rc != hipSuccess) return attr_rc;
  const int grid = 8 * a.g * ((a.k_tiles * a.n_tiles + 7) / 8);
  if (grid <= 0) return hipSuccess;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(C::NT), C::LDS_BYTES, s, a);
  return (int)hipGetLastError();
}

}  // namespace rd
