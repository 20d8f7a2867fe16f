/* The specialised attention kernels (attn_fast.h) at head_dim 64 and 128. */
#include "attn_fast.h"

#define TM_PRE_FAST(T, TN, D) \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_pre_fast_##TN##_d##D(TmAttnPreArgs p) { \
    attn_pre_fast<T, D>(p); \
  }
TM_PRE_FAST(bf16_t, bf16, 64)
TM_PRE_FAST(bf16_t, bf16, 128)
TM_PRE_FAST(f16_t, f16, 64)
TM_PRE_FAST(f16_t, f16, 128)

#define TM_BWD_FAST(T, TN, D, CAUSAL, CN)                                                     \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_dq_fast_##TN##_d##D##CN(TmAttnDqArgs p) {                                           \
    __shared__ __align__(1024) char lds[DqLds<D>::BYTES];                                     \
    attn_dq_fast<T, D, CAUSAL>(p, lds, blockIdx.x, gridDim.x);                                \
  }                                                                                           \
  TM_DKDV_FAST(T, TN, D, CAUSAL, CN)
#define TM_DKDV_FAST(T, TN, D, CAUSAL, CN)                                                    \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_dkdv_fast_##TN##_d##D##CN(TmAttnDkdvArgs p) {                                       \
    __shared__ __align__(1024) char lds[Dkdv2wLds<D>::BYTES];                                 \
    attn_dkdv_2w<T, D, CAUSAL>(p, lds, blockIdx.x, gridDim.x);                                \
  }
#define TM_DKDV_1W(T, TN, CAUSAL, CN)                                                         \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_dkdv_fast_##TN##_d64##CN##_1w(    \
      TmAttnDkdvArgs p) {                                                                     \
    attn_dkdv_1w<T, 64, CAUSAL, false>(p);                                                    \
  }
TM_DKDV_1W(bf16_t, bf16, false, )
TM_DKDV_1W(bf16_t, bf16, true, _causal)
TM_DKDV_1W(f16_t, f16, false, )
TM_DKDV_1W(f16_t, f16, true, _causal)
/* Single-pass backward with atomic dQ (opt-in: bwd=atomic): the dK/dV
 * kernel plus dQ = dS K per query block, and the passes around it. */
#define TM_BWD_FUSED(T, TN, D, CAUSAL, CN)                                                    \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_fused_fast_##TN##_d##D##CN(       \
      TmAttnFusedArgs p) {                                                                    \
    attn_dkdv_1w<T, D, CAUSAL, true>(p.kv, p.dq_acc);                                         \
  }
#define TM_BWD_FAST_ALL(T, TN)           \
  TM_BWD_FUSED(T, TN, 64, false, )       \
  TM_BWD_FUSED(T, TN, 64, true, _causal) \
  TM_BWD_FUSED(T, TN, 128, false, )      \
  TM_BWD_FUSED(T, TN, 128, true, _causal) \
  TM_BWD_FAST(T, TN, 64, false, )        \
  TM_BWD_FAST(T, TN, 64, true, _causal)  \
  TM_BWD_FAST(T, TN, 128, false, )       \
  TM_BWD_FAST(T, TN, 128, true, _causal)
TM_BWD_FAST_ALL(bf16_t, bf16)
TM_BWD_FAST_ALL(f16_t, f16)

#define TM_FWD_FAST(T, TN, D, CAUSAL, CN)                                                     \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void  \
  tm_attn_fwd_fast_##TN##_d##D##CN(TmAttnFwdArgs p) {                                         \
    attn_fwd_fast<T, D, CAUSAL>(p);                                                           \
  }
#define TM_FWD_FAST_ALL(T, TN)           \
  TM_FWD_FAST(T, TN, 64, false, )        \
  TM_FWD_FAST(T, TN, 64, true, _causal)  \
  TM_FWD_FAST(T, TN, 128, false, )       \
  TM_FWD_FAST(T, TN, 128, true, _causal)
TM_FWD_FAST_ALL(bf16_t, bf16)
TM_FWD_FAST_ALL(f16_t, f16)

/* dq_acc = 0 (count a multiple of 4), before the fused backward */
extern "C" __global__ __launch_bounds__(256) void tm_attn_dq_acc_zero(TmAttnDqAccArgs p) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i < p.count) *(f32x4 *)(p.acc + i) = (f32x4){0.f, 0.f, 0.f, 0.f};
}

#define TM_DQ_CONVERT(T, TN, D) \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_dq_convert_##TN##_d##D(TmAttnDqAccArgs p) { \
    attn_dq_convert<T, D>(p); \
  }
TM_DQ_CONVERT(bf16_t, bf16, 64)
TM_DQ_CONVERT(bf16_t, bf16, 128)
TM_DQ_CONVERT(f16_t, f16, 64)
TM_DQ_CONVERT(f16_t, f16, 128)
