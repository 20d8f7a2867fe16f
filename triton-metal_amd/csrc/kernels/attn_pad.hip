/*
 * The 16-bit attention kernels (attn_fast.h, PAD) at head dimensions other than
 * 64 and 128: multiples of 8 up to 128, contracted at the next of 32, 64, 80, 96
 * and 128 columns.  They carry the generic kernels' numerics (fp32 row sums of
 * the unrounded P) on the 16-bit MFMAs, which run 16 times the fp32 ones'
 * rate: at bf16, causal, 32 heads of 1000 rows, head_dim 80 the forward went
 * from 251 to 21.8 us, dQ from 285 to 24.1, dK/dV from 561 to 35.0.  What bounds
 * them is what bounds attn_fast.h's kernels, plus the columns between head_dim
 * and the contracted width (scores contract whole 32-column steps: 96 for 80).
 * f16 holds P unscaled (PBias in attn_fast.h).  dQ and dK/dV of few heads run over
 * ranges (attn_ranges.hip); the forward does not.
 */
#include "attn_fast.h"

#define TM_PAD_ONE(T, TN, D, DC, CAUSAL, CN)                                                  \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_fwd_generic_##TN##_p##DC##CN(TmAttnFwdArgs p) {                                     \
    attn_fwd_fast<T, D, CAUSAL, DC, true>(p);                                                 \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_dq_generic_##TN##_p##DC##CN(TmAttnDqArgs p) {                                       \
    __shared__ __align__(1024) char lds[DqLds<D>::BYTES];                                     \
    attn_dq_fast<T, D, CAUSAL, DC, true>(p, lds, blockIdx.x, gridDim.x);                      \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_dkdv_generic_##TN##_p##DC##CN(TmAttnDkdvArgs p) {                                   \
    __shared__ __align__(1024) char lds[Dkdv2wLds<D>::BYTES];                                 \
    attn_dkdv_2w<T, D, CAUSAL, DC, true>(p, lds, blockIdx.x, gridDim.x);                      \
  }
#define TM_PAD_WIDTH(T, TN, D, DC)        \
  TM_PAD_ONE(T, TN, D, DC, false, )       \
  TM_PAD_ONE(T, TN, D, DC, true, _causal)
#define TM_PAD_ALL(T, TN)                                                                       \
  TM_PAD_WIDTH(T, TN, 64, 32)                                                                   \
  TM_PAD_WIDTH(T, TN, 64, 64)                                                                   \
  TM_PAD_WIDTH(T, TN, 128, 80)                                                                  \
  TM_PAD_WIDTH(T, TN, 128, 96)                                                                  \
  TM_PAD_WIDTH(T, TN, 128, 128)                                                                 \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_pre_generic_##TN##_p64(TmAttnPreArgs p) { \
    attn_pre_fast<T, 64, true>(p);                                                              \
  }                                                                                             \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_pre_generic_##TN##_p128(TmAttnPreArgs p) { \
    attn_pre_fast<T, 128, true>(p);                                                             \
  }
TM_PAD_ALL(bf16_t, bf16)
TM_PAD_ALL(f16_t, f16)
