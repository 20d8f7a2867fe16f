/*
 * 16-bit GEMMs whose rows start at any 2-byte address (odd leading dimensions),
 * row-major or with one operand stored transposed: gemm_fast.h's ragged kernels
 * with register-staged tiles (UNAL).  tm_{gemm,sae}_generic_* are the 64 x 64-tile
 * ones of every layout, and the fp32-MFMA kernel (gemm_generic.h) for strides
 * that are not unit in either dimension: TmGemmArgs.layout says which.
 * (Operands whose buffers have no 14 bytes behind them stay on that too.)
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

static_assert((GENERIC_A + GENERIC_B) * 4 <= TM_GEMM_GROUP_LDS && group_lds(64) == TM_GEMM_GROUP_LDS, "shared LDS");

#define TM_GEMM_UNAL(NAME, T, EPI, TILE, BT, AT)                                              \
  extern "C" __global__ __launch_bounds__(TILE * 2) void NAME(TmGemmArgs p) {                 \
    __shared__ __align__(1024) char lds[group_lds(TILE)];                                     \
    gemm_fast<T, EPI, true, TILE, TILE, BT, AT, 1, false, true>(p, tiles_at<TILE>(lds));                      \
  }
/* 64 x 64 tiles with K ranges across workgroups */
#define TM_GEMM_UNAL_KS(NAME, T, BT, AT, KG)                                                  \
  extern "C" __global__ __launch_bounds__(128 * KG) void NAME(TmGemmArgs p) {                 \
    __shared__ __align__(1024) char lds[KG * group_lds(64)];                                  \
    gemm_fast<T, EPI_NONE, true, 64, 64, BT, AT, KG, true, true>(p, tiles_at<64>(lds));       \
  }
#define TM_GEMM_UNAL_ALL(T, TN)                                                               \
  TM_GEMM_UNAL(tm_gemm_unaligned_##TN, T, EPI_NONE, 256, false, false)                       \
  TM_GEMM_UNAL(tm_gemm_unaligned_nt_##TN, T, EPI_NONE, 256, true, false)                     \
  TM_GEMM_UNAL(tm_sae_unaligned_##TN, T, EPI_BIAS_RELU, 256, false, false)                   \
  TM_GEMM_UNAL(tm_gemm_unaligned_t128_##TN, T, EPI_NONE, 128, false, false)                  \
  TM_GEMM_UNAL(tm_gemm_unaligned_nt_t128_##TN, T, EPI_NONE, 128, true, false)                \
  TM_GEMM_UNAL(tm_gemm_unaligned_tn_t128_##TN, T, EPI_NONE, 128, false, true)                \
  TM_GEMM_UNAL(tm_sae_unaligned_t128_##TN, T, EPI_BIAS_RELU, 128, false, false)              \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_t64_ks_##TN, T, false, false, 1)                          \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_t64_k4_ks_##TN, T, false, false, 4)                       \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_nt_t64_ks_##TN, T, true, false, 1)                        \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_nt_t64_k4_ks_##TN, T, true, false, 4)                     \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_tn_t64_ks_##TN, T, false, true, 1)                        \
  TM_GEMM_UNAL_KS(tm_gemm_unaligned_tn_t64_k4_ks_##TN, T, false, true, 4)                     \
  extern "C" __global__ __launch_bounds__(512) void tm_gemm_generic_##TN(TmGemmArgs p) {      \
    extern __shared__ __align__(1024) char lds[];                                             \
    switch (p.layout) {                                                                       \
      case TM_GEMM_NN: gemm_groups<T, EPI_NONE, true, 64, false, false, true>(p, tiles_at<64>(lds)); break; \
      case TM_GEMM_NT: gemm_groups<T, EPI_NONE, true, 64, true, false, true>(p, tiles_at<64>(lds)); break;  \
      case TM_GEMM_TN: gemm_groups<T, EPI_NONE, true, 64, false, true, true>(p, tiles_at<64>(lds)); break;  \
      default: gemm_generic<T, EPI_NONE>(p, (float *)lds, (float *)lds + GENERIC_A);          \
    }                                                                                         \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(512) void tm_sae_generic_##TN(TmGemmArgs p) {       \
    extern __shared__ __align__(1024) char lds[];                                             \
    if (p.layout == TM_GEMM_NN) gemm_groups<T, EPI_BIAS_RELU, true, 64, false, false, true>(p, tiles_at<64>(lds)); \
    else gemm_generic<T, EPI_BIAS_RELU>(p, (float *)lds, (float *)lds + GENERIC_A);           \
  }
TM_GEMM_UNAL_ALL(bf16_t, bf16)
TM_GEMM_UNAL_ALL(f16_t, f16)
