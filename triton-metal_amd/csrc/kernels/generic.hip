/*
 * Generic gfx950 kernels for the dense hot path: arbitrary strides, ragged
 * shapes, any head dimension up to 128, causal or not.  They stage tiles through
 * LDS as f32 and contract on v_mfma_f32_16x16x4_f32, which multiplies exactly
 * for all three element types (gemm_generic.h, attn_generic.h).  What runs here:
 * 16-bit attention whose rows are not 16-byte aligned, whose head dimension is
 * no multiple of 8, or whose grid is tiny, and the forward of one long head of few
 * columns (ranges fill the chip); fp32 products of at most two 32-wide steps of K,
 * of strides that are not 1, or of ragged sizes whose 16-byte loads have no room
 * behind an operand; the range combines and reduces; Delta; fp32 attention of part
 * of 32 columns where attn_x3.hip, whose fallback these bodies are, is slower.  The
 * reference's numerics:
 *   - f32 accumulation everywhere (GEMMKernel.swift:46, AttentionKernel.swift:59-65);
 *   - P and dS rounded to the element type before the dot they feed
 *     (AttentionKernel.swift:59-65, AttentionBackwardKernel.swift:155-160, :357-369);
 *   - exp2 with sm_scale folded into log2(e) (AttentionKernel.swift:79-80);
 *   - the log2-unit row statistic L = m + log2(l) (AttentionKernel.swift:33-39).
 */
#include "attn_generic.h"
#include "gemm_generic.h"

/* The forward's key-range partials combined (TmAttnFwdArgs.part): for each
 * row, m = max_s m_s, l = sum_s 2^(m_s - m) l_s, O = sum_s 2^(m_s - m) O_s / l,
 * L = m + log2(l) -- the online softmax's own rescaling, applied across the
 * ranges.  Ranges with l_s = 0 (every key masked for the row) add nothing.
 * 64 threads per row (head_dim up to 128), 4 rows per workgroup. */
template <typename T>
TM_DEV void attn_fwd_combine(const TmAttnFwdArgs &p) {
  constexpr int SMAX = 16; /* the planner's largest split */
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n = p.n_ctx, D = p.head_dim, S = p.splits;
  if (row >= (int64_t)p.heads * n) return;
  const int bh = (int)(row / n), q = (int)(row - (int64_t)bh * n);
  const int lane = threadIdx.x & 63;
  const int64_t range = (int64_t)p.heads * n; /* rows per range */
  const float *pml = p.part + (int64_t)S * range * D;
  /* every range's (m, l), then every range's two O values, each as one batch
   * of independent loads */
  float m_s[SMAX], l_s[SMAX];
#pragma unroll
  for (int s = 0; s < SMAX; ++s) {
    const bool in = s < S;
    m_s[s] = in ? pml[(s * range + row) * 2] : 0.f;
    l_s[s] = in ? pml[(s * range + row) * 2 + 1] : 0.f;
  }
  float o0_s[SMAX], o1_s[SMAX];
#pragma unroll
  for (int s = 0; s < SMAX; ++s) {
    const float *po = p.part + (s * range + row) * D;
    o0_s[s] = s < S && lane < D ? po[lane] : 0.f;
    o1_s[s] = s < S && lane + 64 < D ? po[lane + 64] : 0.f;
  }
  float m = TM_NEG_INF;
#pragma unroll
  for (int s = 0; s < SMAX; ++s)
    if (l_s[s] > 0.f) m = fmaxf(m, m_s[s]);
  float l = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
  for (int s = 0; s < SMAX; ++s) {
    if (!(l_s[s] > 0.f)) continue;
    const float w = exp2f(m_s[s] - m);
    l += w * l_s[s];
    o0 += w * o0_s[s];
    o1 += w * o1_s[s];
  }
  const float inv = 1.f / l;
  T *O = (T *)p.o + (int64_t)bh * p.stride_head + (int64_t)q * p.stride_seq;
  if (lane < D) O[lane] = from_f32<T>(o0 * inv);
  if (lane + 64 < D) O[lane + 64] = from_f32<T>(o1 * inv);
  if (p.lse && lane == 0) p.lse[(int64_t)bh * p.stride_lse + q] = m + log2f(l);
}

/* ---------------------------------------------------------------------------
 * attn_bwd_preprocess: Delta_i = sum_d dO_id * O_id in f32
 * (AttentionBackwardKernel.swift:53-136).  64 rows per workgroup, 16 per
 * wave: 16 lanes share a row (lane l sums d = l % 16 + 16 j), four rows at a
 * time with all their loads issued together, then a 16-lane reduction.
 * ------------------------------------------------------------------------- */
template <typename T>
TM_DEV void attn_pre_generic(const TmAttnPreArgs &p) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int bh = blockIdx.y;
  const int64_t base = (int64_t)bh * p.stride_head;
  const T *O = (const T *)p.o + base;
  const T *dO = (const T *)p.dout + base;
  const int sub = lane & 15, grp = lane >> 4;
#pragma unroll
  for (int it = 0; it < 4; ++it) {
    const int row = blockIdx.x * 64 + wave * 16 + it * 4 + grp;
    float acc = 0.f;
    if (row < p.n_ctx) {
#pragma unroll
      for (int j = 0; j < 8; ++j) { /* head_dim <= 128 */
        const int d = sub + 16 * j;
        if (d < p.head_dim) {
          const int64_t off = (int64_t)row * p.stride_seq + d;
          acc += to_f32(O[off]) * to_f32(dO[off]);
        }
      }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (sub == 0 && row < p.n_ctx) p.delta[(int64_t)bh * p.stride_lse + row] = acc;
  }
}

/* The backward's range partials summed (TmAttnSplitReduceArgs): one row of
 * each output per 64 lanes (head_dim up to 128), 4 rows per workgroup, every
 * range's values loaded as one batch. */
template <typename T>
TM_DEV void attn_split_reduce(const TmAttnSplitReduceArgs &p) {
  constexpr int SMAX = 16; /* the planner's largest split */
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int n = p.n_ctx, D = p.head_dim, S = p.splits;
  if (row >= (int64_t)p.heads * n) return;
  const int bh = (int)(row / n), q = (int)(row - (int64_t)bh * n);
  const int lane = threadIdx.x & 63;
  const int64_t plane = (int64_t)p.heads * n * D;
  for (int w = 0; w < p.outputs; ++w) {
    float v0[SMAX], v1[SMAX];
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      const float *src = p.part + (int64_t)(s * p.outputs + w) * plane + row * D;
      v0[s] = s < S && lane < D ? src[lane] : 0.f;
      v1[s] = s < S && lane + 64 < D ? src[lane + 64] : 0.f;
    }
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      a0 += v0[s];
      a1 += v1[s];
    }
    const float scale = w ? p.scale1 : p.scale0;
    T *out = (T *)(w ? p.out1 : p.out0) + (int64_t)bh * p.stride_head + (int64_t)q * p.stride_seq;
    if (lane < D) out[lane] = from_f32<T>(a0 * scale);
    if (lane + 64 < D) out[lane + 64] = from_f32<T>(a1 * scale);
  }
}

/* ---------------------------------------------------------------------------
 * tm_probe: one MFMA against the identity plus a plain store; out[i] == i for
 * i < 256 on a working device (the reference's probe idea, Runtime.swift:125-178).
 * ------------------------------------------------------------------------- */
extern "C" __global__ __launch_bounds__(64) void tm_probe(float *out) {
  const int l = threadIdx.x, g = l >> 4, c = l & 15;
  bf16x8 a, b;
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int k = 8 * g + s;
    a[s] = (bf16_t)(c == k ? 1.f : 0.f);
    b[s] = (bf16_t)(k < 16 ? (float)(k * 16 + c) : 0.f);
  }
  f32x4 d = mfma_16x16x32(a, b, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
  for (int r = 0; r < 4; ++r) out[(4 * g + r) * 16 + c] = d[r];
}

/* ---- named instantiations (the symbols the runtime looks up) -------------- */

#define TM_GEMM(T, NAME, SAE_NAME) \
  extern "C" __global__ __launch_bounds__(256) void NAME(TmGemmArgs p) {                     \
    __shared__ float a_lds[GENERIC_A], b_lds[GENERIC_B];                                      \
    gemm_generic<T, EPI_NONE>(p, a_lds, b_lds);                                               \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) void SAE_NAME(TmGemmArgs p) {                 \
    __shared__ float a_lds[GENERIC_A], b_lds[GENERIC_B];                                      \
    gemm_generic<T, EPI_BIAS_RELU>(p, a_lds, b_lds);                                          \
  }
TM_GEMM(float, tm_gemm_generic_f32, tm_sae_generic_f32)

#define TM_FWD_COMBINE(T, TN)                                                                  \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_fwd_combine_##TN(TmAttnFwdArgs p) {  \
    attn_fwd_combine<T>(p);                                                                    \
  }
TM_FWD_COMBINE(float, f32)
TM_FWD_COMBINE(f16_t, f16)
TM_FWD_COMBINE(bf16_t, bf16)

#define TM_SPLIT_REDUCE(T, TN)                                                                  \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_split_reduce_##TN(                   \
      TmAttnSplitReduceArgs p) {                                                                \
    attn_split_reduce<T>(p);                                                                    \
  }
TM_SPLIT_REDUCE(float, f32)
TM_SPLIT_REDUCE(f16_t, f16)
TM_SPLIT_REDUCE(bf16_t, bf16)

#define TM_PRE(T, NAME) \
  extern "C" __global__ __launch_bounds__(256) void NAME(TmAttnPreArgs p) { attn_pre_generic<T>(p); }
TM_PRE(float, tm_attn_pre_generic_f32)
TM_PRE(f16_t, tm_attn_pre_generic_f16)
TM_PRE(bf16_t, tm_attn_pre_generic_bf16)

#define TM_ATTN_FWD(T, TN, DP, CAUSAL, CN)                                                    \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_fwd_generic_##TN##_d##DP##CN(     \
      TmAttnFwdArgs p) {                                                                      \
    __shared__ __align__(16) float k[generic_tile(DP)], v[generic_tile(DP)];                  \
    attn_fwd_generic<T, DP, CAUSAL>(p, k, v);                                                 \
  }
#define TM_ATTN_DQ(T, TN, DP, CAUSAL, CN)                                                     \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_dq_generic_##TN##_d##DP##CN(      \
      TmAttnDqArgs p) {                                                                       \
    __shared__ float k[32 * (DP + 1)], v[32 * (DP + 1)];                                      \
    attn_dq_generic<T, DP, CAUSAL>(p, k, v);                                                  \
  }
#define TM_ATTN_DKDV(T, TN, DP, CAUSAL, CN)                                                   \
  extern "C" __global__ __launch_bounds__(256) void tm_attn_dkdv_generic_##TN##_d##DP##CN(    \
      TmAttnDkdvArgs p) {                                                                     \
    __shared__ float q[32 * (DP + 1)], d[32 * (DP + 1)], l[32], dl[32];                       \
    attn_dkdv_generic<T, DP, CAUSAL>(p, q, d, l, dl);                                         \
  }
#define TM_ATTN_ONE(T, TN, DP, CAUSAL, CN) \
  TM_ATTN_FWD(T, TN, DP, CAUSAL, CN)       \
  TM_ATTN_DQ(T, TN, DP, CAUSAL, CN)        \
  TM_ATTN_DKDV(T, TN, DP, CAUSAL, CN)
#define TM_ATTN_DT(T, TN, DP)        \
  TM_ATTN_ONE(T, TN, DP, false, )    \
  TM_ATTN_ONE(T, TN, DP, true, _causal)
#define TM_ATTN_ALL_DP(T, TN) \
  TM_ATTN_DT(T, TN, 32)       \
  TM_ATTN_DT(T, TN, 64)       \
  TM_ATTN_DT(T, TN, 96)       \
  TM_ATTN_DT(T, TN, 128)
TM_ATTN_ALL_DP(f16_t, f16)
TM_ATTN_ALL_DP(bf16_t, bf16)
/* fp32 on the fp32 MFMAs, beside attn_x3.hip's: the head dimensions and problem
 * sizes that the planner keeps here (attn_fp32_mfma in runtime.cpp) */
#define TM_ATTN_MFMA32(NAME, DP)                   \
  TM_ATTN_##NAME(float, f32, DP, false, _mfma32)   \
  TM_ATTN_##NAME(float, f32, DP, true, _causal_mfma32)
TM_ATTN_MFMA32(FWD, 32)
TM_ATTN_MFMA32(FWD, 64)
TM_ATTN_MFMA32(FWD, 96)
TM_ATTN_MFMA32(FWD, 128)
TM_ATTN_MFMA32(DQ, 32)
TM_ATTN_MFMA32(DQ, 64)
TM_ATTN_MFMA32(DKDV, 32)
TM_ATTN_MFMA32(DKDV, 64)
TM_ATTN_MFMA32(DKDV, 128)
