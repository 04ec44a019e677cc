// Four-wave GEMM core for launches that do not fill the device: tiles of 128 or 64 rows, HBM -> LDS by direct loads as in
// rd_gemm_dlds.h, a 2 x 2 grid of waves.
//
// What bounds such a launch is the time of one tile, a chain of slabs.  The plain ring of rd_gemm_dlds.h reads a slab's first
// fragments behind the slab's barrier and the rest one substep ahead, and with two or four matrix-core instructions a substep
// nothing covers the LDS round trips; the ping-pong schedule pays two barriers a slab.  Here a slab's fragments are all in
// registers before its first matrix-core instruction: while the wave multiplies slab t it reads every fragment of slab t + 1
// and requests slab t + S, spread evenly over the matrix-core instructions, and there is one barrier a slab.
//
//   slab t: MFMAs on register set t & 1 | fragments of slab t + 1 -> set (t + 1) & 1 | loads of slab t + S into slab t's slot,
//           whose fragments all left it during slab t - 1
//   end:    own share of slab t + 2 landed, own LDS reads returned; barrier
//
// us, the best of the other cores | this one: 512 x 4096 x 4096 in 2 groups 60 | 32, 2048 x 2048 x 2048 in 4 39 | 28, trans_rhs
// 36 | 28; trans_rhs 259 x 10432 x 336 in 3 134 | 24; tgmm 13785 x 960 x 400 in 24 (skewed) 82 | 41.  On launches of more than a
// round of 256 x 256 tiles it moves more bytes through LDS per product than those and is behind (small_tile_variant() in
// rd_capi.hip has the lines).
//
// STREAMS: a kernel whose tiles read the weights of groups of one row tile past the caches (gmm_kernel).
#pragma once
#include "rd_gemm_dlds.h"

namespace rd {

template <int BM_, int BN_, int BK_, bool A_KMAJOR_, bool B_KMAJOR_, int STAGES_, bool HALF_ = false, bool STREAMS_ = false>
struct WsCfg {
  typedef bf16_bits Elem;  // 16 bits per element: bf16, or float16 with HALF
  static constexpr bool F32 = false, WS = true, HALF = HALF_, STREAMS = STREAMS_;
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WAVES_M = 2, WAVES_N = 2, STAGES = STAGES_;
  static constexpr bool A_KMAJOR = A_KMAJOR_, B_KMAJOR = B_KMAJOR_, VEC = true, DLDS = true, PINGPONG = false, MIXED = false,
                        SPLITK = true;
  static constexpr int NW = 4, NT = 256;
  static constexpr int WM = BM / 2, WN = BN / 2;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static constexpr int KSTEPS = BK / 16;
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int EPI_PITCH = WN * 2 + 16;
  static constexpr int EPI_BYTES = NW * WM * EPI_PITCH;
  static constexpr int RING_BYTES = STAGES * STAGE_BYTES;
  static constexpr int LDS_BYTES = RING_BYTES > EPI_BYTES ? RING_BYTES : EPI_BYTES;
  static constexpr int WAVES_PER_EU = LDS_BYTES <= 80 * 1024 ? 2 : 1;  // work-groups of four waves that share a compute unit
  static_assert(BM % 64 == 0 && BN % 64 == 0, "tile shape");
  static_assert(STAGES >= 3, "ring depth");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");
};

template <class C, class = void>
struct IsWs { static constexpr bool value = false; };
template <class C>
struct IsWs<C, decltype((void)C::WS)> { static constexpr bool value = true; };

namespace ws_detail {
template <int V>
struct Int { static constexpr int value = V; };
}  // namespace ws_detail

template <class C, bool LIVE, int B_AUX>
__device__ __forceinline__ void ws_kloop(const bf16_bits* __restrict__ Ap, int lda, int a_lim,
                                         const bf16_bits* __restrict__ Bp, int ldb, int b_lim, int klen,
                                         unsigned char* smem, int wave, int lane, f32x16_t (&acc)[C::TM][C::TN]) {
  const int wm = wave >> 1, wn = wave & 1;
  constexpr int S = C::STAGES;
  typedef DldsLoader<C::BM, C::BK, C::NW, C::A_KMAJOR> LdA;
  typedef DldsLoader<C::BN, C::BK, C::NW, C::B_KMAJOR, B_AUX> LdB;
  LdA la; LdB lb;
  la.init(Ap, lda, a_lim, klen, wave, lane);
  lb.init(Bp, ldb, b_lim, klen, wave, lane);
  DldsFragReader<C::BM, C::BK, C::TM, C::A_KMAJOR> fra;
  DldsFragReader<C::BN, C::BK, C::TN, C::B_KMAJOR> frb;
  fra.init(wm * C::WM, lane);
  frb.init(wn * C::WN, lane);

  const int nk = (klen + C::BK - 1) / C::BK;
  constexpr int PA = LdA::PER, PB = LdB::PER, L = PA + PB;  // loads a wave issues per slab
  constexpr int FR = C::TM + C::TN;             // fragments per 16-wide substep
  constexpr int R = FR * C::KSTEPS;             // fragments per slab
  constexpr int MF = C::TM * C::TN * C::KSTEPS; // MFMAs per slab
  static_assert((S - 2) * L < 64, "vmcnt is 6 bits");

  auto issue_one = [&](int step, int slot_off, int q, auto full_tag) {
    const int k0 = step * C::BK;
    const bool tail = decltype(full_tag)::value == 0 && k0 + C::BK > klen;
    if (q < PA) {
      __amdgpu_buffer_rsrc_t r = la.resource();
      if (tail) la.template issue<true>(r, smem + slot_off, wave, q, k0, klen);
      else la.template issue<false>(r, smem + slot_off, wave, q, k0, klen);
    } else {
      __amdgpu_buffer_rsrc_t r = lb.resource();
      if (tail) lb.template issue<true>(r, smem + slot_off + C::A_BYTES, wave, q - PA, k0, klen);
      else lb.template issue<false>(r, smem + slot_off + C::A_BYTES, wave, q - PA, k0, klen);
    }
  };

  bf16x8_t fa[2][C::KSTEPS][C::TM], fb[2][C::KSTEPS][C::TN];
  auto read_one = [&](auto set_tag, int slot_off, int f) {
    constexpr int SET = decltype(set_tag)::value;
    const unsigned char* ra = smem + slot_off;
    const int ks = f / FR, j = f % FR;
    if (j < C::TM) fa[SET][ks][j] = fra.read(ra, j, ks);
    else fb[SET][ks][j - C::TM] = frb.read(ra + C::A_BYTES, j - C::TM, ks);
  };

  // prologue: the whole ring requested, slab 0's fragments in registers, slab 1 in LDS
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nk) {
#pragma unroll
      for (int q = 0; q < L; ++q) issue_one(s, s * C::STAGE_BYTES, q, ws_detail::Int<0>{});
      la.advance(); lb.advance();
    }
  if (S <= nk) wait_vmcnt<(S - 1) * L < 63 ? (S - 1) * L : 63>(); else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  if (LIVE) {
#pragma unroll
    for (int f = 0; f < R; ++f) read_one(ws_detail::Int<0>{}, 0, f);
  }
  if (S <= nk) wait_vmcnt<(S - 2) * L>(); else wait_vmcnt<0>();
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();

  int cur = 0;  // byte offset of slab t's slot
  auto slab = [&](int t, auto set_tag, auto steady_tag) {
    constexpr int SET = decltype(set_tag)::value;
    constexpr bool STEADY = decltype(steady_tag)::value != 0;
    const int next_off = cur == (S - 1) * C::STAGE_BYTES ? 0 : cur + C::STAGE_BYTES;
    const bool next = STEADY || t + 1 < nk, more = STEADY || t + S < nk;
    constexpr int OPS = R + L;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
#pragma unroll
      for (int o = m * OPS / MF; o < (m + 1) * OPS / MF; ++o) {
        // op o: loads and reads interleaved evenly
        const int lo = o * L / OPS, hi = (o + 1) * L / OPS;
        if (hi > lo) { if (more) issue_one(t + S, cur, lo, steady_tag); }
        else if (LIVE && next) read_one(ws_detail::Int<1 - SET>{}, next_off, o - lo);
      }
      const int ks = m / (C::TM * C::TN), ij = m % (C::TM * C::TN);
      if (LIVE) acc[ij / C::TN][ij % C::TN] = mfma_32x32x16<C::HALF>(fb[SET][ks][ij % C::TN], fa[SET][ks][ij / C::TN], acc[ij / C::TN][ij % C::TN]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) { la.advance(); lb.advance(); }
    if (more) wait_vmcnt<(S - 2) * L>(); else wait_vmcnt<0>();
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    cur = next_off;
  };

  const int n_steady = (klen / C::BK - S) & ~1;  // slabs t with (t + S + 1) * BK <= klen, an even count
  int t = 0;
  for (; t < n_steady; t += 2) {
    slab(t, ws_detail::Int<0>{}, ws_detail::Int<1>{});
    slab(t + 1, ws_detail::Int<1>{}, ws_detail::Int<1>{});
  }
  for (; t < nk; t += 2) {
    slab(t, ws_detail::Int<0>{}, ws_detail::Int<0>{});
    if (t + 1 < nk) slab(t + 1, ws_detail::Int<1>{}, ws_detail::Int<0>{});
  }
}

// B_AUX: cache policy of the B operand's loads, as in rd_gemm_dlds.h
template <class C, int B_AUX = 0>
__device__ __forceinline__ void gemm_tile_ws(const bf16_bits* __restrict__ Ap, int lda, int a_lim,
                                             const bf16_bits* __restrict__ Bp, int ldb, int b_lim, int klen,
                                             bf16_bits* __restrict__ Op, int ldo, bf16_bits* smem_,
                                             const SplitK& sk = SplitK()) {
  unsigned char* smem = reinterpret_cast<unsigned char*>(smem_);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const bool patch_live = wm * C::WM < a_lim && wn * C::WN < b_lim;
  f32x16_t acc[C::TM][C::TN];
#pragma unroll
  for (int i = 0; i < C::TM; ++i)
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  if (patch_live) ws_kloop<C, true, B_AUX>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc);
  else ws_kloop<C, false, B_AUX>(Ap, lda, a_lim, Bp, ldb, b_lim, klen, smem, wave, lane, acc);
  if (!splitk_combine<C>(acc, sk, tid, smem)) return;
  store_accumulators<C>(acc, wm, wn, wave, lane, a_lim, b_lim, Op, ldo, smem, sk.edge_lines);
}

}  // namespace rd
