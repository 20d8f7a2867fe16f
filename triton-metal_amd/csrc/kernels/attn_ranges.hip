/*
 * The 16-bit dQ and dK/dV kernels (attn_fast.h) over ranges of their walk: few
 * heads leave most of the chip idle while a workgroup walks thousands of rows in
 * series, so grid z gives each workgroup one of `splits` ranges of its key (query)
 * blocks and tm_attn_split_reduce_* sums the fp32 partials (unrounded, so the
 * result is rounded once, as without ranges).  What bounds them: the serial walk of
 * a range, then the reduce dispatch (3-5 us).  Measured (bf16, dQ + dK/dV, us,
 * without and with): 64 columns 1 head x 4000 rows 144 and 51, 2 x 4096 146 and 71;
 * 128 columns causal 1 x 4000 238 and 69, 8 x 1024 73 and 53; 80 columns causal
 * 1 x 4000 191 and 48.
 */
#include "attn_fast.h"

#define TM_RANGES(T, TN, D, DC, PAD, NAME, CAUSAL, CN)                                        \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void   \
  tm_attn_dq_##NAME##CN##_ranges(TmAttnDqArgs p) {                                            \
    __shared__ __align__(1024) char lds[DqLds<D>::BYTES];                                     \
    attn_dq_fast<T, D, CAUSAL, DC, PAD, true>(p, lds, blockIdx.x, gridDim.x);                 \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void   \
  tm_attn_dkdv_##NAME##CN##_ranges(TmAttnDkdvArgs p) {                                        \
    __shared__ __align__(1024) char lds[Dkdv2wLds<D>::BYTES];                                 \
    attn_dkdv_2w<T, D, CAUSAL, DC, PAD, true>(p, lds, blockIdx.x, gridDim.x);                 \
  }
#define TM_RANGES_BOTH(T, TN, D, DC, PAD, NAME)        \
  TM_RANGES(T, TN, D, DC, PAD, NAME, false, )          \
  TM_RANGES(T, TN, D, DC, PAD, NAME, true, _causal)
#define TM_RANGES_ALL(T, TN)                                   \
  TM_RANGES_BOTH(T, TN, 64, 64, false, fast_##TN##_d64)        \
  TM_RANGES_BOTH(T, TN, 128, 128, false, fast_##TN##_d128)     \
  TM_RANGES_BOTH(T, TN, 64, 32, true, generic_##TN##_p32)      \
  TM_RANGES_BOTH(T, TN, 64, 64, true, generic_##TN##_p64)      \
  TM_RANGES_BOTH(T, TN, 128, 80, true, generic_##TN##_p80)     \
  TM_RANGES_BOTH(T, TN, 128, 96, true, generic_##TN##_p96)     \
  TM_RANGES_BOTH(T, TN, 128, 128, true, generic_##TN##_p128)
TM_RANGES_ALL(bf16_t, bf16)
TM_RANGES_ALL(f16_t, f16)
