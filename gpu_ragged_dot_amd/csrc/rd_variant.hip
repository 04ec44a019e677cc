// One compiled tile shape.  Built once per entry of the variant list in the Makefile, with
//   -DRD_BM= -DRD_BN= -DRD_BK= -DRD_WAVES_M= -DRD_WAVES_N= -DRD_VEC= -DRD_NAME= [-DRD_DLDS=1|2|3|4|5 -DRD_STAGES= -DRD_PINGPONG=1
//   -DRD_F32=1|2|3|4]
// and exports a getter rd_variant_<name>() for its TileVariant record that the C-ABI file collects.
#include "rd_kernels.h"

#define RD_CAT2(a, b) a##b
#define RD_CAT(a, b) RD_CAT2(a, b)
#define RD_STR2(a) #a
#define RD_STR(a) RD_STR2(a)

#ifndef RD_DLDS
#define RD_DLDS 0
#endif
#ifndef RD_STAGES
#define RD_STAGES 2
#endif
#ifndef RD_PINGPONG
#define RD_PINGPONG 0
#endif

#ifndef RD_F32
#define RD_F32 0
#endif

#if RD_DLDS == 4 || RD_DLDS == 6
#define RD_ANY_PITCH 1
#if RD_DLDS == 6
#define RD_IS_THREE 1
#else
#define RD_IS_THREE 0
#endif
#undef RD_DLDS
#define RD_DLDS 0
#else
#define RD_ANY_PITCH 0
#endif

namespace rd {
#if RD_ANY_PITCH
// 16-byte pieces at any address through registers (rd_gemm_rs.h): bf16, float16, float32 rounded to bf16, or float32 as it is
#if RD_F32 == 2 || RD_F32 == 1
typedef float RsElem;
#elif RD_F32 == 4
typedef f16_t RsElem;
#else
typedef bf16_bits RsElem;
#endif
typedef RsCfg<RD_BM, RD_BN, /*A K-major*/ true, /*B K-major*/ false, RsElem, RD_VEC != 0, RD_F32 == 1 && !RD_IS_THREE, RD_IS_THREE, RD_WAVES_N> CfgNN;
typedef RsCfg<RD_BM, RD_BN, true, true, RsElem, RD_VEC != 0, RD_F32 == 1 && !RD_IS_THREE, RD_IS_THREE, RD_WAVES_N> CfgNT;
typedef RsCfg<RD_BM, RD_BN, false, false, RsElem, RD_VEC != 0, RD_F32 == 1 && !RD_IS_THREE, RD_IS_THREE, RD_WAVES_N> CfgTN;
#elif RD_F32 == 4 && RD_DLDS == 3
// float16 arrays on the four-wave direct-to-LDS core: the bf16 core's data movement with the float16 instruction
typedef W4Cfg<RD_BM, RD_BN, /*A K-major*/ true, /*B K-major*/ false, RD_STAGES, true> CfgNN;
typedef W4RCfg<RD_BM, RD_BN, true> CfgNT;
typedef W4Cfg<RD_BM, RD_BN, false, false, RD_STAGES, true> CfgTN;
#elif (RD_F32 == 0 || RD_F32 == 4) && RD_DLDS == 5
// the core of rd_gemm_ws.h, bf16 or float16
typedef WsCfg<RD_BM, RD_BN, RD_BK, /*A K-major*/ true, /*B K-major*/ false, RD_STAGES, RD_F32 == 4> CfgNN;
typedef WsCfg<RD_BM, RD_BN, RD_BK, true, true, RD_STAGES, RD_F32 == 4> CfgNT;
typedef WsCfg<RD_BM, RD_BN, RD_BK, false, false, RD_STAGES, RD_F32 == 4> CfgTN;
// ... and with the weights of short groups streamed past the caches: the tiles that the default rules name for such launches
#if RD_BN == 2 * RD_BM
typedef WsCfg<RD_BM, RD_BN, RD_BK, true, false, RD_STAGES, RD_F32 == 4, /*streams*/ true> CfgNNStream;
#define RD_NN_STREAM &rd::launch_gmm<rd::CfgNNStream, false>
#endif
#if RD_BK == 64
typedef WsCfg<RD_BM, RD_BN, RD_BK, true, true, RD_STAGES, RD_F32 == 4, true> CfgNTStream;
#define RD_NT_STREAM &rd::launch_gmm<rd::CfgNTStream, true>
#endif
#elif (RD_F32 == 0 || RD_F32 == 4) && RD_DLDS == 2
// one LDS ring per operand: one K-major operand in 64-wide slabs (3 slots) - the activations in the forward product,
// the weights A[g,n,k] with trans_rhs (measured 1-3 % ahead of giving them to dout) - everything else in 32-wide
// slabs (4 slots); bf16 or float16
typedef PpCfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, 64, 3, 32, 4, RD_F32 == 4> CfgNN;
typedef PpCfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, true, true, 32, 4, 64, 3, RD_F32 == 4> CfgNT;
typedef PpCfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, false, false, 32, 4, 32, 4, RD_F32 == 4> CfgTN;
#elif (RD_F32 == 0 || RD_F32 == 4) && RD_DLDS == 1
typedef DldsCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, RD_STAGES, RD_PINGPONG != 0, 0, RD_F32 == 4> CfgNN;
typedef DldsCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, true, true, RD_STAGES, RD_PINGPONG != 0, 0, RD_F32 == 4> CfgNT;
typedef DldsCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, false, false, RD_STAGES, RD_PINGPONG != 0, 0, RD_F32 == 4> CfgTN;
#elif RD_F32 == 3 && RD_DLDS
// float8 e4m3fn arrays on the float8 matrix-core instruction, direct-to-LDS (rd_gemm_f8.h).  tgmm reads x^T as an
// MN-major operand, whose slab rows span the tile's rows: only for tile heights that are multiples of 256.
typedef F8Cfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, RD_STAGES, 64, 0, /*A K-major*/ true, /*B K-major*/ false, RD_PINGPONG != 0> CfgNN;
typedef F8Cfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, RD_STAGES, 64, 0, true, true, RD_PINGPONG != 0> CfgNT;
#if RD_BM % 256 == 0
typedef F8Cfg<RD_BM, RD_BN, RD_WAVES_M, RD_WAVES_N, RD_STAGES, 64, 0, false, false, RD_PINGPONG != 0> CfgTN;
#else
#define RD_NO_TGMM 1
#endif
#elif RD_F32 == 3
// float8 e4m3fn arrays, widened to bf16 on the way into LDS, bf16 matrix cores, bf16 out
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, RD_VEC != 0, fp8_bits> CfgNN;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, true, true, RD_VEC != 0, fp8_bits> CfgNT;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, false, false, RD_VEC != 0, fp8_bits> CfgTN;
#elif RD_F32 == 4
// float16 arrays on the float16 matrix-core instruction, float16 out
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, RD_VEC != 0, f16_t> CfgNN;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, true, true, RD_VEC != 0, f16_t> CfgNT;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, false, false, RD_VEC != 0, f16_t> CfgTN;
#elif RD_F32 == 2
// float32 arrays, rounded to bf16 on the way into LDS, bf16 matrix cores, float32 out (compute_dtype = bfloat16)
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, RD_VEC != 0, float> CfgNN;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, true, true, RD_VEC != 0, float> CfgNT;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, false, false, RD_VEC != 0, float> CfgTN;
#elif RD_F32
typedef F32Cfg<RD_BM, RD_BN, /*A K-major*/ true, /*B K-major*/ false> CfgNN;
typedef F32Cfg<RD_BM, RD_BN, true, true> CfgNT;
typedef F32Cfg<RD_BM, RD_BN, false, false> CfgTN;
#elif RD_DLDS == 3
typedef W4Cfg<RD_BM, RD_BN, /*A K-major*/ true, /*B K-major*/ false, RD_STAGES> CfgNN;
// both operands K-major: the 64-wide, register-staged form of the core (rd_gemm_w4r.h)
typedef W4RCfg<RD_BM, RD_BN> CfgNT;
typedef W4Cfg<RD_BM, RD_BN, false, false, RD_STAGES> CfgTN;
#else
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, /*A K-major*/ true, /*B K-major*/ false, RD_VEC != 0> CfgNN;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, true, true, RD_VEC != 0> CfgNT;
typedef TileCfg<RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, false, false, RD_VEC != 0> CfgTN;
#endif
}  // namespace rd

#ifndef RD_NN_STREAM
#define RD_NN_STREAM nullptr
#endif
#ifndef RD_NT_STREAM
#define RD_NT_STREAM nullptr
#endif

extern "C" const rd::TileVariant* RD_CAT(rd_variant_, RD_NAME)() {
  static const rd::TileVariant v = {
      RD_STR(RD_NAME), RD_BM, RD_BN, RD_BK, RD_WAVES_M, RD_WAVES_N, RD_VEC, /*dtype: RD_DTYPE_* */ RD_F32, RD_DLDS != 0, RD_STAGES,
      RD_ANY_PITCH, /*splitk*/ RD_ANY_PITCH || (RD_DLDS != 0 && (!RD_F32 || RD_F32 == 3 || RD_F32 == 4)),
      rd::SplitCost<rd::CfgNN>::QUARTERS, rd::SplitCost<rd::CfgNN>::MIN_K, rd::HalvesLastRound<rd::CfgNN>::value ? RD_BN / 2 : RD_BN, rd::SplitsByGain<rd::CfgNN>::value, rd::IsWs<rd::CfgNN>::value, rd::IsMixed<rd::CfgNN>::value,
#ifdef RD_NO_TGMM
      &rd::launch_gmm<rd::CfgNN, false>, &rd::launch_gmm<rd::CfgNT, true>, nullptr,
#else
      &rd::launch_gmm<rd::CfgNN, false>, &rd::launch_gmm<rd::CfgNT, true>, &rd::launch_tgmm<rd::CfgTN>,
#endif
      RD_NN_STREAM, RD_NT_STREAM};
  return &v;
}
