/* The 16-bit GEMM kernels (gemm_fast.h) whose rows of A and B are 16-byte aligned. */
#include "gemm_fast.h"

/* the tiles of one K group in four arrays, and `MORE` for further groups */
#define TM_GEMM_TILES(TILE, MORE)                                                             \
  __shared__ __align__(1024) char tile_a0[TILE * GBK * 2];                                    \
  __shared__ __align__(1024) char tile_b0[TILE * GBK * 2];                                    \
  __shared__ __align__(1024) char tile_a1[TILE * GBK * 2];                                    \
  __shared__ __align__(1024) char tile_b1[TILE * GBK * 2];                                    \
  const GemmTiles<false> tiles = {tile_a0, tile_b0, tile_a1, tile_b1, MORE};

extern "C" __global__ __launch_bounds__(256) void tm_gemm_split_reduce_bf16(TmGemmArgs p) {
  gemm_split_reduce<bf16_t>(p);
}
extern "C" __global__ __launch_bounds__(256) void tm_gemm_split_reduce_f16(TmGemmArgs p) {
  gemm_split_reduce<f16_t>(p);
}

#define TM_GEMM_ONE(NAME, T, EPI, RAGGED, TILE, BT, AT)                                       \
  extern "C" __global__ __launch_bounds__(TILE * 2) void NAME(TmGemmArgs p) {                 \
    TM_GEMM_TILES(TILE, nullptr)                                                              \
    gemm_fast<T, EPI, RAGGED, TILE, TILE, BT, AT>(p, tiles);                                  \
  }
/* K groups and LDS as launched (ragged 64 x 64 tiles, whole ones with the SAE
 * epilogue) */
#define TM_GEMM_GROUPS(NAME, T, EPI, RAGGED, TILE, BT, AT)                                    \
  extern "C" __global__ __launch_bounds__(512) void NAME(TmGemmArgs p) {                      \
    extern __shared__ __align__(1024) char more[];                                            \
    TM_GEMM_TILES(TILE, more)                                                                 \
    gemm_groups<T, EPI, RAGGED, TILE, BT, AT, false>(p, tiles);                               \
  }
/* the 64 x 64-tile GEMMs with K ranges across workgroups ("_ks") */
#define TM_GEMM_KS(NAME, T, RAGGED, BT, AT, KG)                                               \
  extern "C" __global__ __launch_bounds__(128 * KG) void NAME(TmGemmArgs p) {                 \
    if constexpr (KG == 1) {                                                                  \
      TM_GEMM_TILES(64, nullptr)                                                              \
      gemm_fast<T, EPI_NONE, RAGGED, 64, 64, BT, AT, 1, true>(p, tiles);                      \
    } else {                                                                                  \
      __shared__ __align__(1024) char lds[KG * group_lds(64)];                                \
      gemm_fast<T, EPI_NONE, RAGGED, 64, 64, BT, AT, KG, true>(p, tiles_at<64>(lds));         \
    }                                                                                         \
  }
#define TM_GEMM_KS_ALL(T, TN)                                                                 \
  TM_GEMM_KS(tm_gemm_ragged_t64_ks_##TN, T, true, false, false, 1)                            \
  TM_GEMM_KS(tm_gemm_ragged_nt_t64_ks_##TN, T, true, true, false, 1)                          \
  TM_GEMM_KS(tm_gemm_ragged_tn_t64_ks_##TN, T, true, false, true, 1)                          \
  TM_GEMM_KS(tm_gemm_ragged_t64_k4_ks_##TN, T, true, false, false, 4)                         \
  TM_GEMM_KS(tm_gemm_ragged_nt_t64_k4_ks_##TN, T, true, true, false, 4)                       \
  TM_GEMM_KS(tm_gemm_ragged_tn_t64_k4_ks_##TN, T, true, false, true, 4)                       \
  TM_GEMM_KS(tm_gemm_fast_t64_k4_ks_##TN, T, false, false, false, 4)                          \
  TM_GEMM_KS(tm_gemm_fast_nt_t64_k4_ks_##TN, T, false, true, false, 4)                        \
  TM_GEMM_KS(tm_gemm_fast_tn_t64_k4_ks_##TN, T, false, false, true, 4)
TM_GEMM_KS_ALL(bf16_t, bf16)
TM_GEMM_KS_ALL(f16_t, f16)
/* whole 128 x 128 (64 x 64) tiles, the K loop over 2 (2 or 4) wave groups */
#define TM_GEMM_KG(NAME, T, EPI, TILE, BT, AT, KG)                                            \
  extern "C" __global__ __launch_bounds__(2 * TILE * KG) void NAME(TmGemmArgs p) {            \
    __shared__ __align__(1024) char lds[KG * group_lds(TILE)];                                \
    gemm_fast<T, EPI, false, TILE, TILE, BT, AT, KG>(p, tiles_at<TILE>(lds));                 \
  }
#define TM_GEMM_KG_LAYOUT(T, TN, FAMILY, EPI, BT, AT)                                         \
  TM_GEMM_KG(FAMILY##_t128_k2_##TN, T, EPI, 128, BT, AT, 2)                                  \
  TM_GEMM_KG(FAMILY##_t64_k2_##TN, T, EPI, 64, BT, AT, 2)                                    \
  TM_GEMM_KG(FAMILY##_t64_k4_##TN, T, EPI, 64, BT, AT, 4)
#define TM_GEMM_KSPLIT(T, TN)                                                                 \
  TM_GEMM_KG_LAYOUT(T, TN, tm_gemm_fast, EPI_NONE, false, false)                              \
  TM_GEMM_KG_LAYOUT(T, TN, tm_gemm_fast_nt, EPI_NONE, true, false)                            \
  TM_GEMM_KG_LAYOUT(T, TN, tm_gemm_fast_tn, EPI_NONE, false, true)
TM_GEMM_KSPLIT(bf16_t, bf16)
TM_GEMM_KSPLIT(f16_t, f16)
#define TM_GEMM_FAST(T, TN)                                                       \
  TM_GEMM_ONE(tm_gemm_fast_##TN, T, EPI_NONE, false, 256, false, false)                      \
  TM_GEMM_ONE(tm_gemm_ragged_##TN, T, EPI_NONE, true, 256, false, false)                     \
  TM_GEMM_ONE(tm_sae_fast_##TN, T, EPI_BIAS_RELU, false, 256, false, false)                  \
  TM_GEMM_ONE(tm_sae_ragged_##TN, T, EPI_BIAS_RELU, true, 256, false, false)                 \
  TM_GEMM_ONE(tm_gemm_fast_t128_##TN, T, EPI_NONE, false, 128, false, false)                 \
  TM_GEMM_ONE(tm_gemm_ragged_t128_##TN, T, EPI_NONE, true, 128, false, false)                \
  TM_GEMM_GROUPS(tm_sae_fast_t128_##TN, T, EPI_BIAS_RELU, false, 128, false, false)           \
  TM_GEMM_ONE(tm_sae_fast_t128_g1_##TN, T, EPI_BIAS_RELU, false, 128, false, false)           \
  TM_GEMM_ONE(tm_sae_ragged_t128_##TN, T, EPI_BIAS_RELU, true, 128, false, false)            \
  TM_GEMM_ONE(tm_gemm_fast_nt_##TN, T, EPI_NONE, false, 256, true, false)                    \
  TM_GEMM_ONE(tm_gemm_ragged_nt_##TN, T, EPI_NONE, true, 256, true, false)                   \
  TM_GEMM_ONE(tm_gemm_fast_nt_t128_##TN, T, EPI_NONE, false, 128, true, false)               \
  TM_GEMM_ONE(tm_gemm_ragged_nt_t128_##TN, T, EPI_NONE, true, 128, true, false)              \
  TM_GEMM_ONE(tm_gemm_fast_tn_##TN, T, EPI_NONE, false, 256, false, true)                    \
  TM_GEMM_ONE(tm_gemm_ragged_tn_##TN, T, EPI_NONE, true, 256, false, true)                   \
  TM_GEMM_ONE(tm_gemm_fast_tn_t128_##TN, T, EPI_NONE, false, 128, false, true)               \
  TM_GEMM_ONE(tm_gemm_ragged_tn_t128_##TN, T, EPI_NONE, true, 128, false, true)              \
  TM_GEMM_ONE(tm_gemm_fast_t64_##TN, T, EPI_NONE, false, 64, false, false)                   \
  TM_GEMM_GROUPS(tm_gemm_ragged_t64_##TN, T, EPI_NONE, true, 64, false, false)                \
  TM_GEMM_ONE(tm_gemm_ragged_t64_g1_##TN, T, EPI_NONE, true, 64, false, false)                \
  TM_GEMM_GROUPS(tm_sae_fast_t64_##TN, T, EPI_BIAS_RELU, false, 64, false, false)             \
  TM_GEMM_ONE(tm_sae_fast_t64_g1_##TN, T, EPI_BIAS_RELU, false, 64, false, false)             \
  TM_GEMM_GROUPS(tm_sae_ragged_t64_##TN, T, EPI_BIAS_RELU, true, 64, false, false)            \
  TM_GEMM_ONE(tm_sae_ragged_t64_g1_##TN, T, EPI_BIAS_RELU, true, 64, false, false)            \
  TM_GEMM_ONE(tm_gemm_fast_nt_t64_##TN, T, EPI_NONE, false, 64, true, false)                 \
  TM_GEMM_GROUPS(tm_gemm_ragged_nt_t64_##TN, T, EPI_NONE, true, 64, true, false)              \
  TM_GEMM_ONE(tm_gemm_ragged_nt_t64_g1_##TN, T, EPI_NONE, true, 64, true, false)              \
  TM_GEMM_ONE(tm_gemm_fast_tn_t64_##TN, T, EPI_NONE, false, 64, false, true)                 \
  TM_GEMM_GROUPS(tm_gemm_ragged_tn_t64_##TN, T, EPI_NONE, true, 64, false, true)              \
  TM_GEMM_ONE(tm_gemm_ragged_tn_t64_g1_##TN, T, EPI_NONE, true, 64, false, true)              
TM_GEMM_FAST(bf16_t, bf16)
TM_GEMM_FAST(f16_t, f16)
