// GEMM core for operands that cannot be loaded straight into LDS: row pitches that are no multiple of 16 bytes
// (bf16 and float16), float32 arrays that are rounded to bf16 on the way (compute_dtype = bfloat16), and float32 arrays of
// any pitch multiplied to float32's accuracy.  A 256 x 256 tile held by a 2 x 2 grid of waves, 128 x 128 per wave, as in
// rd_gemm_w4.h, or a smaller tile, several work-groups to a compute unit, or 2 x 4 waves on a 128 x 256 tile; HBM -> registers
// -> LDS as in rd_gemm_w4r.h, for any of the four operand layouts.
//
// What bounds it: with the 64 x 64 and 128 x 128 tiles of rd_gemm_tile.h these products were bound by their loads - one
// element per instruction where the pitch is odd, one slab in flight where the source is float32 - at 40-85 and 300-430
// TFLOP/s (bf16 8191 x 2047 x 4095 in 16 groups, fwd / dlhs / drhs: 2300 / 3080 / 1620 us; float32 8192 x 4096 x 4096 in
// 8: 683 / 668 / 899).  Here: 218 / 271 / 337 and 387 / 397 / 371 us; aligned bf16 16384 x 4096 x 4096 in 8 groups 574 us
// (960 TFLOP/s).  Left over: the latency of the first slabs and of the epilogue, which nothing else on the compute unit
// hides under a 256 x 256 tile (one round of them, 4096^3 float32: 146 us, 940 TFLOP/s), the last, partly filled round, and
// pieces that straddle cache lines (20-50 % against the same sizes aligned).  How:
//  * a load is always 16 bytes per lane (a "piece"), at whatever address the element has: global memory takes 16-byte
//    accesses at any alignment.  Every 8 lanes (K-major) or every 32 / 64 (MN-major) read consecutive memory;
//  * a slab is 128 bytes of every K-major row (64 bf16 or 32 float32 contraction indices), 16 pieces per lane for both
//    operands, and two slabs are in flight in registers beside the two in LDS (bf16: 2 x 64 KB, float32 rounded: 2 x 32 KB);
//  * 128 x 256 on eight waves: three quarters of the 128 x 128 tile's loads, and two waves on a SIMD (fills_rounds_128x256() in rd_capi.hip);
//  * float32 rounded to bf16: 256 x 256 on eight waves of 128 x 64, whose second wave on a SIMD multiplies while the first converts and
//    writes: 0.98 times the four waves' time in gmm (1144 random calls at 16-byte pitches; 803 at others 0.99), 0.94 in tgmm (163);
//  * the pieces are converted and written to LDS, and their registers refilled, spread evenly over the gaps between the
//    matrix-core instructions of a slab.
// float32 multiplied as float32 (FULL) is bound by its matrix-core instruction, 157 TFLOP/s at most, of which this core reaches 86-92 %
// (4096 x 4096 x 3072: 766 / 733 / 713 us).  So float32 goes through the bf16 matrix cores, 16 times as fast, as three bf16 terms a number
// (THREE): x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1) holds all 24 bits, and of the nine products
// of two numbers' terms the three left out (x1 y2, x2 y1, x2 y2: |x1| <= 2^-8 |x|, |x2| <= 2^-17 |x|) come to at most 2^-24 of the whole one,
// what one rounding of float32 may cost, and to a fifth of that as a root mean square.
//  * The terms are made on the way into LDS, which holds three planes of a slab in the bf16 layout, and all three of a
//    fragment are read per substep: 24 matrix-core instructions per 12 fragments (128 x 256 tile, eight waves of 64 x 64), half the
//    fragment reads of a bf16 product.  A piece's way takes 28 vector instructions, in seven steps spread over the gaps between matrix-core
//    instructions; eight waves, two on a SIMD, keep the matrix cores busy 77 % of a work-group's time (profiles/any_pitch_core.md).
//  * 16384 x 4096 x 2048 in one group, tgmm: 1274 us (216 TFLOP/s, i.e. 1294 on the bf16 matrix cores; 881 us on zeros), FULL on
//    128 x 128 tiles 1879; 8192 x 2048 x 2048 in 16 softmax-sized groups, fwd / dlhs / drhs: 377 / 378 / 380, FULL 574 / 594 / 595.
//    Power bounds it, as it does the bf16 products.
//  * The error against sums in float64 is 0.83-0.87 of FULL's (16 products are added up per rounding, two there): relative 2-norm on N(0, 1) data
//    2.4e-7 (FULL 2.9e-7) for 256 products, 6.8e-7 (8.0e-7) for 2048; over 90 random sizes never above FULL's, nor where products are
//    subnormal.  Of one and two products it would be: see kFewProducts.
//  * Where the terms do not hold a number, the tile is computed again by FULL (kThreeLeast).
// One loop serves all slabs.  Where a load goes is a clamped offset from a base; on the slab that holds the last contraction
// index the base, the offset and its limit change (enter_last), so that no load touches memory outside the operand's rows,
// and from there on what is not the operand's is cut off on the way into LDS (trim).  A second loop for those slabs, with
// loads of their own, had the compiler spill 300 registers under two MN-major operands (float32 tgmm, 8192 x 4096 x 4096 in 8
// groups: 499 us so, 371 without; 16384 x 2048 x 2048 in 32: 408 and 266).
#pragma once
#include <type_traits>
#include "rd_gemm_dlds.h"

namespace rd {

// Src: bf16_bits, f16_t, or float (float32 out).  FULL: float32 stays float32 on its way through LDS and is multiplied by
// v_mfma_f32_32x32x2_f32; THREE: it becomes three bf16 terms; otherwise it is rounded to bf16.  VEC: k and n are multiples of 8 (float32: of 4), so that no piece
// crosses the end of a row and the last slab needs no shifting.
template <int BM_, int BN_, bool A_KMAJOR_, bool B_KMAJOR_, typename Src, bool VEC_, bool FULL_ = false, bool THREE_ = false, int WAVES_N_ = 2>
struct RsCfg {
  typedef Src Elem;
  static constexpr bool F32 = false, RS = true, HALF = std::is_same<Src, f16_t>::value;
  static constexpr int BM = BM_, BN = BN_, BK = 128 / (int)sizeof(Src), WAVES_M = 2, WAVES_N = WAVES_N_, STAGES = 2;
  static constexpr bool A_KMAJOR = A_KMAJOR_, B_KMAJOR = B_KMAJOR_, VEC = VEC_, DLDS = false, PINGPONG = false, MIXED = false,
                        SPLITK = true;
  static constexpr int NW = WAVES_M * WAVES_N, NT = 64 * NW;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr bool FULL = FULL_, THREE = THREE_;
  static constexpr int LB = FULL ? 4 : 2;                  // bytes of an element (THREE: of each of its terms) in LDS
  static constexpr int TERMS = THREE ? 3 : 1;
  static constexpr int KMF = FULL ? 4 : THREE ? 6 : 1;     // matrix-core instructions per block and substep
  static constexpr int KSTEPS = FULL ? BK / 8 : BK / 16;   // substeps per slab
  // work-groups per compute unit
  static constexpr int WAVES_PER_EU = NW == 8 ? 2 : THREE ? (BM * BN < 128 * 128 ? 2 : 1) : BM * BN > 128 * 128 ? 1 : BM * BN < 128 * 128 ? 3 : 2;
  static constexpr int A_TERM = BM * BK * LB, B_TERM = BN * BK * LB;         // one term of a slab in LDS
  static constexpr int A_BYTES = TERMS * A_TERM, B_BYTES = TERMS * B_TERM;  // one slab in LDS
  static constexpr int SLOT_BYTES = A_BYTES + B_BYTES;
  static constexpr int EPI_PITCH = WN * 2 + 16;
  static constexpr int EPI_BYTES = sizeof(Src) == 2 ? NW * WM * EPI_PITCH : 0;
  static constexpr int RING_BYTES = 2 * SLOT_BYTES;
  static constexpr int LDS_BYTES = RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES;
  static_assert(FULL || THREE ? BM % 64 == 0 && BN % 64 == 0 : BM % (A_KMAJOR ? 64 : 128) == 0 && BN % 128 == 0, "tile shape");
  static_assert(!(FULL && THREE) && (!(FULL || THREE) || std::is_same<Src, float>::value), "float32 only");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

template <class C, class = void>
struct IsRs { static constexpr bool value = false; };
template <class C>
struct IsRs<C, decltype((void)C::RS)> { static constexpr bool value = true; };

// The 128-bit value v shifted down by `bytes` (0 .. 16, whole elements), zeros from above.
__device__ __forceinline__ u32x4_t shift_down(u32x4_t v, int bytes) {
  uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
  if (bytes >= 8) { lo = hi; hi = 0; bytes -= 8; }
  if (bytes >= 8) { lo = 0; bytes = 0; }
  const int b = bytes * 8;
  lo = (lo >> b) | (b ? hi << (64 - b) : 0);
  hi >>= b;
  return u32x4_t{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// One operand's slab, [T rows][BK] (K-major) or [BK][T columns] (MN-major), in pieces of 16 bytes: which memory each lane
// reads for each of its pieces, and where the piece goes in LDS (the layout DldsFragReader reads).
template <int T, int BK, int NW, bool KMAJOR, typename Src, bool VEC, int LB = 2>
struct RsLoader {
  static constexpr int EPP = 16 / (int)sizeof(Src);              // elements per piece
  static constexpr int PPR = (KMAJOR ? BK : T) / EPP;            // pieces per slab row
  static constexpr int RPI = 64 / PPR;                           // slab rows per wave-wide load
  static constexpr int PER = (KMAJOR ? T : BK) / RPI / NW;       // pieces per lane
  static constexpr int LDS_ROW = (KMAJOR ? BK : T) * LB;         // bytes of a slab row in LDS
  static constexpr int LDS_STEP = NW * RPI * LDS_ROW;            // from one of a lane's pieces to its next
  static_assert(PPR <= 64 && 64 % PPR == 0 && (KMAJOR ? T : BK) % (RPI * NW) == 0, "slab does not split evenly");
  // the chunk permutation of DldsFragReader repeats from one of a lane's pieces to the next
  static_assert(KMAJOR ? (NW * RPI) % 16 == 0 : (NW * RPI) % (LB == 4 ? 8 : 4) == 0, "chunk permutation");

  const Src* base;   // first element of the current slab (one piece before it once the slab holds the last contraction index)
  long long step;    // elements from one slab to the next
  uint32_t off0;     // byte offset of piece 0 from base; piece j lies j * row_step further, but no further than off_last
  uint32_t row_step, off_last;
  int ld, lim, klen;
  int slab, last;    // index of the current slab; of the slab that holds the last contraction index
  int lds;           // byte of piece 0 in the operand's region of a slot

  static __host__ __device__ __forceinline__ int slab_row(int wave, int lane, int j) { return wave * RPI + lane / PPR + j * NW * RPI; }

  __host__ __device__ __forceinline__ void init(const Src* p, int ld_, int lim_, int klen_, int wave, int lane) {
    base = p; ld = ld_; lim = lim_; klen = klen_;
    step = KMAJOR ? BK : (long long)BK * ld;
    slab = 0; last = (klen - 1) / BK;
    const int row0 = slab_row(wave, lane, 0), piece = lane % PPR;
    // rows past the tile's limit re-read its last row, columns past it the last piece that holds one of the tile's:
    // what they hold never reaches a stored element.  (An MN-major piece may run past the end of its row, at most into the
    // row behind it, which exists: the slab ends before the last contraction index.)
    const int e = KMAJOR ? piece * EPP : imin(piece * EPP, (lim - 1) / EPP * EPP);
    off_last = KMAJOR ? ((uint32_t)(lim - 1) * (uint32_t)ld + (uint32_t)e) * (uint32_t)sizeof(Src) : ~0u;
    off0 = ((uint32_t)row0 * (uint32_t)ld + (uint32_t)e) * (uint32_t)sizeof(Src);
    row_step = (uint32_t)(NW * RPI * sizeof(Src)) * (uint32_t)ld;
    const int chunk = sizeof(Src) == LB ? piece : piece >> 1;  // 16-byte chunk of the LDS row; a rounded float32 piece fills half of one
    const int c = KMAJOR ? (LDS_ROW == 128 ? chunk ^ ((row0 >> 1) & 7) : chunk ^ ((row0 >> 2) & 3))
                : LB == 4 ? chunk ^ (((row0 >> 2) & 1) << 3) : chunk ^ ((row0 & (T >= 128 ? 3 : T / 32 - 1)) << 2);
    lds = row0 * LDS_ROW + (c << 4) + (sizeof(Src) == LB ? 0 : (piece & 1) * 8);
    if (last == 0) enter_last(wave, lane);
  }

  // The slab that holds the last contraction index.  A piece that would run past the contraction length (K-major) or past
  // the tile's columns (MN-major) is read from before them instead, rows past the contraction length re-read its last one;
  // trim() takes out what is not the operand's.  The place may lie before the slab's first element (the row it is read
  // along holds a whole piece up to there): offsets count from one piece before it.
  __host__ __device__ __forceinline__ int last_at(int lane) const {
    const int e = lane % PPR * EPP;
    return KMAJOR ? imin(e, klen - EPP - last * BK) : imin(e, lim - EPP);
  }
  __host__ __device__ __forceinline__ void enter_last(int wave, int lane) {
    const uint32_t at = (uint32_t)(last_at(lane) + EPP);
    const int rows = KMAJOR ? lim : klen - last * BK;
    base -= EPP;
    off0 = ((uint32_t)slab_row(wave, lane, 0) * (uint32_t)ld + at) * (uint32_t)sizeof(Src);
    off_last = ((uint32_t)(rows - 1) * (uint32_t)ld + at) * (uint32_t)sizeof(Src);
  }
  // On to the next slab; behind the last one the loads stay where they are (and trim() leaves only zeros).
  __host__ __device__ __forceinline__ void next(int wave, int lane) {
    ++slab;
    if (slab <= last) base += step;
    if (slab == last) enter_last(wave, lane);
  }
  __host__ __device__ __forceinline__ uint32_t offset(int j) const {
    const uint32_t o = off0 + (uint32_t)j * row_step;
    return o > off_last ? off_last : o;
  }
  __device__ __forceinline__ u32x4_t fetch(int j) const { return load_any<u32x4_t>(reinterpret_cast<const unsigned char*>(base) + offset(j)); }
  // By how many elements piece j of slab `at_slab` (the last one or behind it) has to come down; EPP or more: all zeros.
  __host__ __device__ __forceinline__ int surplus(int wave, int lane, int j, int at_slab) const {
    const bool gone = at_slab > last || (!KMAJOR && slab_row(wave, lane, j) >= klen - last * BK);
    return gone ? EPP : lane % PPR * EPP - last_at(lane);
  }
  __device__ __forceinline__ u32x4_t trim(int wave, int lane, int j, int at_slab, u32x4_t v) const {
    const int shift = surplus(wave, lane, j, at_slab);
    if constexpr (VEC) return shift == 0 ? v : u32x4_t{0, 0, 0, 0};
    else return shift_down(v, imin(shift, EPP) * (int)sizeof(Src));
  }
  __device__ __forceinline__ void commit(unsigned char* region, int j, u32x4_t v) const {
    unsigned char* d = region + lds + j * LDS_STEP;
    if constexpr (sizeof(Src) == LB) {
      *reinterpret_cast<u32x4_t*>(d) = v;
    } else {
      const f32x4_t f = __builtin_bit_cast(f32x4_t, v);
      *reinterpret_cast<u32x2_t*>(d) = u32x2_t{pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])};
    }
  }
  __device__ __forceinline__ void put(unsigned char* region, int j, u32x2_t v) const {
    *reinterpret_cast<u32x2_t*>(region + lds + j * LDS_STEP) = v;
  }
  // The new base and the lane's offset are opaque to the compiler: it would otherwise carry an address per piece through
  // the loop, and there are no registers for those.
  __device__ __forceinline__ void advance(int wave, int lane) {
    next(wave, lane);
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    base = reinterpret_cast<const Src*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b) |
                                        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32));
    asm volatile("" : "+v"(off0));
  }
};

// Fragments of float32 slabs (FULL), 8 contraction indices at a time: lane l feeds row / column (l & 31) of a block with the
// four indices 4 (l >> 5) .. + 3, one per matrix-core instruction - that instruction multiplies two indices, one per half
// wave, and since both operands name the same two it does not matter that they are not neighbours.  K-major rows give the
// four in one 16-byte read, MN-major slabs in four reads of 32 consecutive columns.
template <int T, int TILES, bool KMAJOR>
struct RsFullFrag {
  int addr[KMAJOR ? 4 : 1];
  __device__ __forceinline__ void init(int idx0, int lane) {
    const int h = lane >> 5;
    if (KMAJOR) {
      const int r = lane & 31;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) addr[ks] = (idx0 + r) * 128 + (((2 * ks + h) ^ ((r >> 1) & 7)) << 4);
    } else {
      // rows 8 ks + 4 h + e have bit 2 equal to h: their 32-column halves of 64 are exchanged where it is set
      addr[0] = 4 * h * T * 4 + (((idx0 + (lane & 31)) * 4) ^ (h << 7));
    }
  }
  __device__ __forceinline__ f32x4_t read(const unsigned char* region, int tile, int ks) const {
    if (KMAJOR) {
      return *reinterpret_cast<const f32x4_t*>(region + addr[ks] + tile * 32 * 128);
    } else {
      // a block's 32 columns are one half of an aligned 64: the next block is the other half
      const unsigned char* p = region + (addr[0] ^ ((tile & 1) << 7)) + (tile >> 1) * 256 + ks * 8 * T * 4;
      f32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const float*>(p + e * T * 4);
      return v;
    }
  }
};
template <class C, int T, int TILES, bool KMAJOR>
struct RsFrag {
  typedef typename std::conditional<C::FULL, RsFullFrag<T, TILES, KMAJOR>, DldsFragReader<T, C::BK, TILES, KMAJOR>>::type type;
};

// THREE multiplies exactly what FULL multiplies only where the terms hold the whole number, 24 bits: not below 2^-110, where the third
// one's last bit leaves bf16 (2^-133), and not for infinities, NaN and what rounds to infinity.  The least magnitude seen on
// the way into LDS (as bits << 1, less one: zeros come out on top) tells the former, a sum that is no finite number the
// latter; a tile that has either is computed again by FULL.
constexpr uint32_t kThreeLeast = ((127u - 110u) << 24) - 1u;
// A product alone is rounded once there, and the products of terms left out come on top of that here (up to half of the last bit: rows of a
// group 1, 2, 3, 4, 16: 2-norm error in units of 2^-24 0.58 | 0.42, 0.56 | 0.52, 0.55 | 0.60, 0.54 | 0.67, 0.56 | 1.24, THREE | FULL).  So
// contractions of at most this many indices, tgmm over groups of one and two rows, are multiplied as float32 (rs_few_products()).
constexpr int kFewProducts = 2;
__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) { return a < b ? a : b; }

namespace rs_detail {
template <int V>
struct Int { static constexpr int value = V; };
}  // namespace rs_detail

// Slab t lives in LDS slot t & 1 and, before that, in register set t & 1.  The pieces of slab t + 1 are written to LDS
// during the substeps of slab t (16 contraction indices each, fragments read one substep ahead), except that the last
// substep, which follows the slab's barrier, already writes the first pieces of slab t + 2 into the slot slab t has left.
// Each write is followed by the load of the same piece two slabs further on.  float32 slabs have half as many substeps
// for as many pieces, so a gap there carries a write and a load where a 16-bit slab alternates them.
template <class C, bool LIVE>
__device__ __forceinline__ void rs_kloop(const typename C::Elem* __restrict__ Ap, int lda, int a_lim,
                                         const typename C::Elem* __restrict__ Bp, int ldb, int b_lim, int klen,
                                         unsigned char* smem, int wave, int lane, f32x16_t (&acc)[C::TM][C::TN], uint32_t& least) {
  typedef typename C::Elem E;
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  typedef RsLoader<C::BM, C::BK, C::NW, C::A_KMAJOR, E, C::VEC, C::LB> LdA;
  typedef RsLoader<C::BN, C::BK, C::NW, C::B_KMAJOR, E, C::VEC, C::LB> LdB;
  LdA la; LdB lb;
  la.init(Ap, lda, a_lim, klen, wave, lane);
  lb.init(Bp, ldb, b_lim, klen, wave, lane);
  typename RsFrag<C, C::BM, C::TM, C::A_KMAJOR>::type fra;
  typename RsFrag<C, C::BN, C::TN, C::B_KMAJOR>::type frb;
  auto read_a = [&](const unsigned char* region, int r, int ks) { return fra.read(region + r / C::TM * C::A_TERM, r % C::TM, ks); };
  auto read_b = [&](const unsigned char* region, int r, int ks) { return frb.read(region + r / C::TN * C::B_TERM, r % C::TN, ks); };
  fra.init(wm * C::WM, lane);
  frb.init(wn * C::WN, lane);

  const int nk = (klen + C::BK - 1) / C::BK;  // the last slab, nk - 1, holds the last contraction index
  constexpr int PA = LdA::PER, PB = LdB::PER, P = PA + PB;
  constexpr int RA = C::TM * C::TERMS, RB = C::TN * C::TERMS;  // fragments per substep
  constexpr int MF = C::TM * C::TN * C::KMF, R0 = RA + RB;
  // pieces moved per substep: the last one, which follows the slab's barrier, takes pieces 0 .. HEAD - 1 (of the slab after
  // next), substep u of the others pieces part(u + 1) .. part(u + 2) - 1
  constexpr auto part = [](int u) constexpr { return u * P / C::KSTEPS; };
  constexpr int HEAD = part(1), MOST = (P + C::KSTEPS - 1) / C::KSTEPS;
  // What the gaps between a substep's matrix-core instructions carry.  Large patches: one fragment read each in the first
  // ones, then the pieces, spread out (a write and the load that refills its registers in one gap or in two).  Small
  // patches have fewer gaps than reads and pieces: every gap carries its share of both.
  constexpr bool ROOMY = !C::THREE && MF - R0 >= MOST;
  constexpr int GAP = MF - R0 >= 2 * MOST ? 2 : 1;

  u32x4_t regs[2][P];
  auto fetch_one = [&](auto set_tag, int q) {
    constexpr int SET = decltype(set_tag)::value;
    regs[SET][q] = q < PA ? la.fetch(q) : lb.fetch(q - PA);
  };
  // THREE: step st of a piece's way into LDS - its first term, what that leaves, the second term, what that leaves, the third -
  // a few vector instructions each, for one gap between two matrix-core instructions.
  constexpr int kThreeSteps = 7;
  u32x2_t term;
  auto three_step = [&](auto set_tag, int slot_off, int q, int st) {
    constexpr int SET = decltype(set_tag)::value;
    u32x4_t& r = regs[SET][q];
    auto f = [&](int e) { const uint32_t w = r[e]; return __builtin_bit_cast(float, w); };
    auto leave = [&](int h) {  // elements 2 h and 2 h + 1 minus their term: exact
      r[2 * h] = __builtin_bit_cast(uint32_t, f(2 * h) - __builtin_bit_cast(float, term[h] << 16));
      r[2 * h + 1] = __builtin_bit_cast(uint32_t, f(2 * h + 1) - __builtin_bit_cast(float, term[h] & 0xffff0000u));
    };
    auto note = [&](int h) { least = umin(least, umin((r[2 * h] << 1) - 1u, (r[2 * h + 1] << 1) - 1u)); };
    if (st % 3 == 0) {
      term = u32x2_t{pack_bf16x2(f(0), f(1)), pack_bf16x2(f(2), f(3))};
      if (q < PA) la.put(smem + slot_off + st / 3 * C::A_TERM, q, term);
      else lb.put(smem + slot_off + C::A_BYTES + st / 3 * C::B_TERM, q - PA, term);
      if (st == 0) note(0);
    } else {
      if (st == 1) note(1);
      leave(st % 3 - 1);
    }
  };
  auto commit_one = [&](auto set_tag, int slot_off, int q) {
    constexpr int SET = decltype(set_tag)::value;
    if constexpr (C::THREE) {
#pragma unroll
      for (int st = 0; st < kThreeSteps; ++st) three_step(set_tag, slot_off, q, st);
    } else if (q < PA) la.commit(smem + slot_off, q, regs[SET][q]);
    else lb.commit(smem + slot_off + C::A_BYTES, q - PA, regs[SET][q]);
  };
  // Before pieces first .. first + count - 1 of slab `step` are written: where that slab holds the last contraction index or
  // lies behind it, take out what is not the operand's.
  auto trim_some = [&](auto set_tag, int step, int first, int count) {
    constexpr int SET = decltype(set_tag)::value;
    if (step >= nk - 1) {
#pragma unroll
      for (int q = first; q < first + count; ++q)
        regs[SET][q] = q < PA ? la.trim(wave, lane, q, step, regs[SET][q]) : lb.trim(wave, lane, q - PA, step, regs[SET][q]);
    }
  };
  auto advance = [&]() { la.advance(wave, lane); lb.advance(wave, lane); };

  // slab 0 through the registers into LDS, slab 1 in registers with its first pieces written, slab 2 requested
  auto prologue = [&]() {
#pragma unroll
    for (int q = 0; q < P; ++q) fetch_one(rs_detail::Int<0>{}, q);
    advance();
#pragma unroll
    for (int q = 0; q < P; ++q) fetch_one(rs_detail::Int<1>{}, q);
    advance();
    trim_some(rs_detail::Int<0>{}, 0, 0, P);
#pragma unroll
    for (int q = 0; q < P; ++q) commit_one(rs_detail::Int<0>{}, 0, q);
#pragma unroll
    for (int q = 0; q < P; ++q) fetch_one(rs_detail::Int<0>{}, q);
    advance();
    trim_some(rs_detail::Int<1>{}, 1, 0, HEAD);
#pragma unroll
    for (int q = 0; q < HEAD; ++q) commit_one(rs_detail::Int<1>{}, C::SLOT_BYTES, q);
#pragma unroll
    for (int q = 0; q < HEAD; ++q) fetch_one(rs_detail::Int<1>{}, q);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): slab 0 is written
    __builtin_amdgcn_s_barrier();
  };

  typedef typename std::conditional<C::FULL, f32x4_t, bf16x8_t>::type frag_t;
  frag_t fa[2][RA], fb[2][RB];
  auto first_fragments = [&]() {
    if (LIVE) {
#pragma unroll
      for (int i = 0; i < RA; ++i) fa[0][i] = read_a(smem, i, 0);
#pragma unroll
      for (int j = 0; j < RB; ++j) fb[0][j] = read_b(smem + C::A_BYTES, j, 0);
    }
  };

  auto slab = [&](int t, auto next_tag) {
    constexpr int NEXT = decltype(next_tag)::value;  // (t + 1) & 1
    const int cur_off = (1 - NEXT) * C::SLOT_BYTES, next_off = NEXT * C::SLOT_BYTES;
#pragma unroll
    for (int u = 0; u < C::KSTEPS; ++u) {
      const bool last = u == C::KSTEPS - 1;
      if (last) {  // own reads of slab t returned, own pieces of slab t + 1 written; behind the barrier slab t + 1 is complete
        advance();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      const unsigned char* ra = smem + (last ? next_off : cur_off);  // fragments of the next substep
      const unsigned char* rb = ra + C::A_BYTES;
      const int us = last ? 0 : u + 1;
      const int first = last ? 0 : part(u + 1), count = last ? HEAD : part(u + 2) - part(u + 1);
      if (last) trim_some(rs_detail::Int<1 - NEXT>{}, t + 2, first, count);
      else trim_some(next_tag, t + 1, first, count);
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        const int i = m % (C::TM * C::TN) / C::TN, j = m % C::TN, ke = m / (C::TM * C::TN);
        if (LIVE && ROOMY) {
          if (m < RA) fa[(u + 1) & 1][m] = read_a(ra, m, us);
          else if (m < R0) fb[(u + 1) & 1][m - RA] = read_b(rb, m - RA, us);
        } else if (LIVE) {
#pragma unroll
          for (int r = m * R0 / MF; r < (m + 1) * R0 / MF; ++r) {
            if (r < RA) fa[(u + 1) & 1][r] = read_a(ra, r, us);
            else fb[(u + 1) & 1][r - RA] = read_b(rb, r - RA, us);
          }
        }
        auto write = [&](int p) {
          if (last) commit_one(rs_detail::Int<1 - NEXT>{}, cur_off, p);  // of slab t + 2
          else commit_one(next_tag, next_off, first + p);                // of slab t + 1
        };
        auto load = [&](int p) {
          if (last) fetch_one(rs_detail::Int<1 - NEXT>{}, p);  // of slab t + 4
          else fetch_one(next_tag, first + p);                 // of slab t + 3
        };
        if constexpr (ROOMY) {
          const int p = (m - R0) / GAP;
          if (m >= R0 && p < count) {
            if ((m - R0) % GAP == 0) write(p);
            if ((m - R0) % GAP == GAP - 1) load(p);
          }
        } else if constexpr (C::THREE) {
          constexpr int ST = kThreeSteps + 1;  // the last one is the load
#pragma unroll
          for (int s = m * count * ST / MF; s < (m + 1) * count * ST / MF; ++s) {
            if (s % ST == kThreeSteps) load(s / ST);
            else if (last) three_step(rs_detail::Int<1 - NEXT>{}, cur_off, s / ST, s % ST);
            else three_step(next_tag, next_off, first + s / ST, s % ST);
          }
        } else {
#pragma unroll
          for (int p = m * count / MF; p < (m + 1) * count / MF; ++p) { write(p); load(p); }
        }
        if (LIVE) {
          // float32 results leave straight from the accumulators, a register holding 32 consecutive columns of a row;
          // 16-bit results go through LDS and want four consecutive columns per lane (operands swapped)
          if constexpr (C::FULL) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[u & 1][i][ke], fb[u & 1][j][ke], acc[i][j], 0, 0, 0);
          else if constexpr (C::THREE) {
            // the six products of two terms that are not below the last bit of the whole one, the small ones first
            constexpr int TA[6] = {0, 2, 1, 0, 1, 0}, TB[6] = {2, 0, 1, 1, 0, 0};
            acc[i][j] = mfma_32x32x16<false>(fa[u & 1][TA[ke] * C::TM + i], fb[u & 1][TB[ke] * C::TN + j], acc[i][j]);
          } else if constexpr (sizeof(E) == 2) acc[i][j] = mfma_32x32x16<C::HALF>(fb[u & 1][j], fa[u & 1][i], acc[i][j]);
          else acc[i][j] = mfma_32x32x16<false>(fa[u & 1][i], fb[u & 1][j], acc[i][j]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  prologue();
  first_fragments();
  for (int t = 0; t < nk; t += 2) {  // (an odd nk multiplies one slab of zeros)
    slab(t, rs_detail::Int<1>{});
    slab(t + 1, rs_detail::Int<0>{});
  }

  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();  // the slots are no longer read by any wave
}

// 16-bit results: each wave turns its patch through LDS into rows and stores 16 bytes per lane at whatever address the
// row has; the piece that crosses the tile's last column goes element by element.
template <class C>
__device__ __forceinline__ void rs_store16(const f32x16_t (&acc)[C::TM][C::TN], int wm, int wn, int wave, int lane, int a_lim,
                                           int b_lim, typename C::Elem* __restrict__ Op, int ldo, unsigned char* smem) {
  unsigned char* st = smem + wave * (C::WM * C::EPI_PITCH);
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int row = i * 32 + (lane & 31), col = j * 32 + 8 * g + 4 * (lane >> 5);
        u32x2_t w;
        w[0] = pack_out_x2<C::HALF>(acc[i][j][4 * g + 0], acc[i][j][4 * g + 1]);
        w[1] = pack_out_x2<C::HALF>(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        *reinterpret_cast<u32x2_t*>(st + row * C::EPI_PITCH + col * 2) = w;
      }
  constexpr int CPR = C::WN / 8, ROWS_PER = 64 / CPR, NIT = C::WM / ROWS_PER, BATCH = NIT < 8 ? NIT : NIT % 8 == 0 ? 8 : 6;
  static_assert(NIT % BATCH == 0, "whole batches");
  const int chunk = lane % CPR, r0 = lane / CPR;
  const int gcol = wn * C::WN + chunk * 8, live = b_lim - gcol;  // live: the lane's columns inside the tile
#pragma unroll
  for (int t0 = 0; t0 < NIT; t0 += BATCH) {
    u32x4_t v[BATCH];
#pragma unroll
    for (int b = 0; b < BATCH; ++b)
      v[b] = *reinterpret_cast<const u32x4_t*>(st + ((t0 + b) * ROWS_PER + r0) * C::EPI_PITCH + chunk * 16);
#pragma unroll
    for (int b = 0; b < BATCH; ++b) {
      const int grow = wm * C::WM + (t0 + b) * ROWS_PER + r0;
      if (grow >= a_lim || live <= 0) continue;
      unsigned char* d = reinterpret_cast<unsigned char*>(Op + (size_t)grow * ldo + gcol);
      if (live >= 8) store_any(d, v[b]);
      else
#pragma unroll
        for (int e = 0; e < 7; ++e)
          if (e < live) reinterpret_cast<uint16_t*>(d)[e] = (uint16_t)(v[b][e >> 1] >> ((e & 1) * 16));
    }
  }
}

// float32 results: register v of a 32 x 32 block is 32 consecutive columns of row 8 (v >> 2) + 4 (lane >> 5) + (v & 3) - a
// whole 128-byte line per half wave.  Rows and columns past the tile's limits get an offset outside the output's window,
// which the hardware drops.  Nontemporal, as in store_accumulators(); with SplitK::edge_lines plainly, where rows are no whole number of 64-byte halves of
// a line, so that what a half wave stores ends inside two lines and L2 has to put them together (kEdgeLineRows in rd_kernels.h).
template <class C, int POLICY = kCachePolicyStream>
__device__ __forceinline__ void rs_store32(const f32x16_t (&acc)[C::TM][C::TN], int wm, int wn, int lane, int a_lim, int b_lim,
                                           float* __restrict__ Op, int ldo) {
  const int bytes = ((a_lim - 1) * ldo + b_lim) * 4;  // below 2 GiB: checked on the host
  __amdgpu_buffer_rsrc_t orsrc = __builtin_amdgcn_make_buffer_rsrc((void*)Op, 0, __builtin_amdgcn_readfirstlane(bytes), kBufferFlags);
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j) {
      const int col = wn * C::WN + j * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = wm * C::WM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const int off = row < a_lim && col < b_lim ? (row * ldo + col) * 4 : kOobOffset;
        const float f = acc[i][j][v];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, f), orsrc, off, 0, POLICY);
      }
    }
}

// A tgmm tile of one or two rows: a product, and another one added with one rounding, the bits of the float32 matrix-core instruction.
// Bound by its stores.  230 groups of one row among 256 of 16384 rows, k 2048, n 768: 502 us, as slabs of 32 indices on FULL 814, on terms 719.
template <class C, int POLICY>
__device__ __forceinline__ void rs_few_products(const float* __restrict__ Ap, int lda, int a_lim, const float* __restrict__ Bp, int ldb,
                                                int b_lim, int klen, int wm, int wn, int lane, float* __restrict__ Op, int ldo) {
  const float* __restrict__ A1 = Ap + (size_t)(klen - 1) * lda;  // the second row, or the first one again
  const float* __restrict__ B1 = Bp + (size_t)(klen - 1) * ldb;
  float b0[C::TN], b1[C::TN];
#pragma unroll
  for (int j = 0; j < C::TN; ++j) {
    const int col = wn * C::WN + j * 32 + (lane & 31), c = col < b_lim ? col : b_lim - 1;  // (what lies outside is not stored)
    b0[j] = Bp[c]; b1[j] = B1[c];
  }
  f32x16_t acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int row = wm * C::WM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3), r = row < a_lim ? row : a_lim - 1;
      const float a0 = Ap[r], a1 = A1[r];
#pragma unroll
      for (int j = 0; j < C::TN; ++j) {
        const float f = fmaf(a0, b0[j], 0.f);  // (no zero leaves with a sign, as from the matrix cores)
        acc[i][j][v] = klen > 1 ? fmaf(a1, b1[j], f) : f;
      }
    }
  rs_store32<C, POLICY>(acc, wm, wn, lane, a_lim, b_lim, Op, ldo);
}

// Same contract as gemm_tile(), and: the rows the operands are read along hold at least 8 elements (16-bit) or 4
// (float32) up to and including the tile's last one - k >= 8 and n >= 8.
template <class C, bool EDGE_LINES = false>
__device__ __forceinline__ void gemm_tile_rs(const typename C::Elem* __restrict__ Ap, int lda, int a_lim,
                                             const typename C::Elem* __restrict__ Bp, int ldb, int b_lim, int klen,
                                             typename C::Elem* __restrict__ Op, int ldo, unsigned char* smem,
                                             const SplitK& sk = SplitK()) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  const bool patch_live = wm * C::WM < a_lim && wn * C::WN < b_lim;

  if constexpr (C::THREE && !C::A_KMAJOR) {
    if (klen <= kFewProducts) {
      if (EDGE_LINES && sk.edge_lines) rs_few_products<C, 0>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, wm, wn, lane, Op, ldo);
      else rs_few_products<C, kCachePolicyStream>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, wm, wn, lane, Op, ldo);
      return;
    }
  }

  f32x16_t acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  uint32_t least = ~0u;
  if (patch_live) rs_kloop<C, true>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc, least);
  else rs_kloop<C, false>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc, least);

  if constexpr (C::THREE) {
    // Values that the three terms do not hold: see kThreeLeast.  All waves of the work-group must agree, they share the slabs.
    float probe = 0.f;  // NaN once a sum is no finite number
#pragma unroll
    for (int i = 0; i < C::TM; ++i)
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) probe = fmaf(acc[i][j][v], 0.f, probe);
    uint32_t* flags = reinterpret_cast<uint32_t*>(smem);
    if (tid == 0) flags[0] = 0;
    __syncthreads();
    if (least < kThreeLeast || probe != probe) flags[0] = 1;
    __syncthreads();
    const uint32_t any = flags[0];
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane((int)any)) {
      typedef RsCfg<C::BM, C::BN, C::A_KMAJOR, C::B_KMAJOR, typename C::Elem, C::VEC, true, false, C::WAVES_N> Full;
      static_assert(Full::LDS_BYTES <= C::LDS_BYTES && Full::NT == C::NT, "runs in this launch");
#pragma unroll
      for (int i = 0; i < C::TM; ++i)
#pragma unroll
        for (int j = 0; j < C::TN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
      if (patch_live) rs_kloop<Full, true>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc, least);
      else rs_kloop<Full, false>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc, least);
    }
  }

  if (!splitk_combine<C>(acc, sk, tid, smem)) return;
  if constexpr (sizeof(typename C::Elem) == 2) rs_store16<C>(acc, wm, wn, wave, lane, a_lim, b_lim, Op, ldo, smem);
  else if (EDGE_LINES && sk.edge_lines) rs_store32<C, 0>(acc, wm, wn, lane, a_lim, b_lim, Op, ldo);
  else rs_store32<C>(acc, wm, wn, lane, a_lim, b_lim, Op, ldo);
}

// A row tile of a gmm launch with fewer rows than its height: the same routine on the least multiple of 64 that holds them,
// with as many fewer loads, LDS traffic and matrix-core instructions.  False: the tile is to be computed whole.
// (FULL is compiled with tiles of 64 rows only, and as what THREE falls back to.)
template <class C, int ROWS = 64>
__device__ __forceinline__ bool rs_short_tile(const typename C::Elem* __restrict__ Ap, int lda, int rows,
                                              const typename C::Elem* __restrict__ Bp, int ldb, int cols, int klen,
                                              typename C::Elem* __restrict__ Op, int ldo, void* smem, const SplitK& sk) {
  if constexpr (ROWS >= C::BM || C::FULL) {
    return false;
  } else {
    typedef RsCfg<ROWS, C::BN, true, C::B_KMAJOR, typename C::Elem, C::VEC, false, C::THREE, C::WAVES_N> S;
    static_assert(C::A_KMAJOR && S::LDS_BYTES <= C::LDS_BYTES && S::NT == C::NT, "runs in the tall tile's launch");
    if (rows > ROWS) return rs_short_tile<C, ROWS + 64>(Ap, lda, rows, Bp, ldb, cols, klen, Op, ldo, smem, sk);
    gemm_tile_rs<S>(Ap, lda, rows, Bp, ldb, cols, klen, Op, ldo, static_cast<unsigned char*>(smem), sk);
    return true;
  }
}

}  // namespace rd
