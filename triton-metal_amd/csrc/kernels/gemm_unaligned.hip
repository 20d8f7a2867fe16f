/*
 * 16-bit GEMMs whose rows start at any 2-byte address (odd leading dimensions),
 * row-major or with one operand stored transposed: gemm_fast.h's ragged kernels
 * with register-staged tiles (UNAL).  tm_{gemm,sae}_generic_* are the 64 x 64-tile
 * ones of every layout, and the fp32-MFMA kernel (gemm_generic.h) for strides
 * that are not unit in either dimension: TmGemmArgs.layout says which.
 * The fp32-MFMA kernel, which ran all of these before, converts every element
 * and contracts at a sixteenth of the 16-bit rate.  bf16, row-major, us before
 * and now: 2049 x 4097 x 1025 455 and 50, 4097 x 4099 x 4101 3346 and 264 (rows
 * of 4104 elements, copied to LDS directly: 219), 17 x 4099 x 4097 473 and 16.4,
 * 300 x 200 x 100 11.2 and 4.4.  The tile choice is the aligned kernels':
 * 128 x 128 tiles take 54.6, 260 and (3001 x 3003 x 3005) 126 us where 256 x 256
 * take 50.3, 260 and 98.7.
 */
#include "gemm_fast.h"
#include "gemm_generic.h"

static_assert((GENERIC_A + GENERIC_B) * 4 <= unaligned_lds(64), "shared LDS");

#define TM_GEMM_UNAL(NAME, T, EPI, TILE, BT, AT, KS)                                          \
  extern "C" __global__ __launch_bounds__(TILE * 2) void NAME(TmGemmArgs p) {                 \
    __shared__ __align__(1024) char lds[unaligned_lds(TILE)];                                 \
    gemm_fast<T, EPI, true, TILE, TILE, BT, AT, 1, KS, true>(p, lds);                         \
  }
#define TM_GEMM_UNAL_TILE(T, TN, SUFFIX, TILE)                                                \
  TM_GEMM_UNAL(tm_gemm_unaligned##SUFFIX##_##TN, T, EPI_NONE, TILE, false, false, false)      \
  TM_GEMM_UNAL(tm_gemm_unaligned_nt##SUFFIX##_##TN, T, EPI_NONE, TILE, true, false, false)    \
  TM_GEMM_UNAL(tm_sae_unaligned##SUFFIX##_##TN, T, EPI_BIAS_RELU, TILE, false, false, false)
#define TM_GEMM_UNAL_ALL(T, TN)                                                               \
  TM_GEMM_UNAL_TILE(T, TN, , 256)                                                             \
  TM_GEMM_UNAL_TILE(T, TN, _t128, 128)                                                        \
  TM_GEMM_UNAL(tm_gemm_unaligned_tn_t128_##TN, T, EPI_NONE, 128, false, true, false)          \
  TM_GEMM_UNAL(tm_gemm_unaligned_t64_ks_##TN, T, EPI_NONE, 64, false, false, true)            \
  TM_GEMM_UNAL(tm_gemm_unaligned_nt_t64_ks_##TN, T, EPI_NONE, 64, true, false, true)          \
  TM_GEMM_UNAL(tm_gemm_unaligned_tn_t64_ks_##TN, T, EPI_NONE, 64, false, true, true)          \
  extern "C" __global__ __launch_bounds__(256) void tm_gemm_generic_##TN(TmGemmArgs p) {      \
    __shared__ __align__(1024) char lds[unaligned_lds(64)];                                   \
    switch (p.layout) {                                                                       \
      case TM_GEMM_NN: gemm_fast<T, EPI_NONE, true, 64, 64, false, false, 1, false, true>(p, lds); break; \
      case TM_GEMM_NT: gemm_fast<T, EPI_NONE, true, 64, 64, true, false, 1, false, true>(p, lds); break;  \
      case TM_GEMM_TN: gemm_fast<T, EPI_NONE, true, 64, 64, false, true, 1, false, true>(p, lds); break;  \
      default: gemm_generic<T, EPI_NONE>(p, (float *)lds, (float *)lds + GENERIC_A);                                                \
    }                                                                                         \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) void tm_sae_generic_##TN(TmGemmArgs p) {       \
    __shared__ __align__(1024) char lds[unaligned_lds(64)];                                   \
    if (p.layout == TM_GEMM_NN) gemm_fast<T, EPI_BIAS_RELU, true, 64, 64, false, false, 1, false, true>(p, lds); \
    else gemm_generic<T, EPI_BIAS_RELU>(p, (float *)lds, (float *)lds + GENERIC_A);                                                   \
  }
TM_GEMM_UNAL_ALL(bf16_t, bf16)
TM_GEMM_UNAL_ALL(f16_t, f16)
