/*
 * The fp32 attention kernels on the bf16 matrix cores: the generic kernels'
 * work split, ranges and numerics (attn_generic.h) with every product as eight bf16
 * MFMAs of three-way split operands (split3.h), which take half the fp32 MFMA's
 * time and round less often.
 *
 * One 256-thread workgroup takes 64 queries (keys in dK/dV), 16 per wave, held in
 * registers as split operands; it walks blocks of keys (queries), staged through
 * registers -- the next block's loads are in flight behind the current one's
 * MFMAs -- and split once into LDS planes of bf16 rows with attn_fast.h's
 * layout, read by ds_read_b128 and, as the k-major operand, ds_read_b64_tr_b16.
 * Softmax, row sums, P and dS stay fp32; P and dS are split for their products.
 * Measured (us, forward / dQ / dK, dV on the fp32 MFMA and here): 16 heads of 2048
 * rows at 64 columns 204 / 239 / 306 and 172 / 190 / 231, at 128 columns 379 / 478
 * / 669 and 295 / 342 / 569; 2 heads of 96 11.7 / 12.8 / 16.4 and 10.1 / 10.6 /
 * 14.2 (six products, which lost bits: 160 / 168 / 207, 267 / 296 / 466 and 10.0 /
 * 9.9 / 14.1).  The MFMA pipes are busy 34 / 45 / 49% of the time at 64 columns and
 * 39 / 50 / 38% at 128; the rest is the split (5.5 VALU
 * operations an element and as much again for P and dS) and the LDS round trip
 * between a block's two barriers, which two or three workgroups per CU cover
 * in part.
 *
 * A workgroup that meets what the split cannot represent (split3.h) leaves its
 * result and runs the generic kernel's body instead.
 */
#include "attn_fast.h"
#include "attn_generic.h"
#include "split3.h"

namespace {

typedef f32x4 f32x4_any __attribute__((aligned(4)));

constexpr int pitch(int dp) { return dp <= 64 ? 64 : 128; }
/* rows of a block: 64 at DP <= 64, else 32 (LDS, registers) */
constexpr int block_rows(int dp) { return dp <= 64 ? 64 : 32; }
/* bytes of one operand's three planes */
constexpr int planes(int dp) { return 3 * block_rows(dp) * pitch(dp) * 2; }
constexpr int lds_bytes(int dp) {
  return 2 * planes(dp) > 8 * generic_tile(dp) ? 2 * planes(dp) : 8 * generic_tile(dp);
}

/* eight floats of a row from column d, zeros at or past D */
TM_DEV void load8(const float *row, int d, int D, bool in, f32x4 (&v)[2]) {
  if (in && d + 8 <= D) {
    v[0] = *(const f32x4_any *)(row + d);
    v[1] = *(const f32x4_any *)(row + d + 4);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e >> 2][e & 3] = in && d + e < D ? row[d + e] : 0.f;
  }
}

TM_DEV void split_run(const f32x4 (&v)[2], u32x4 (&part)[3]) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = v[e >> 2][e & 3] * X3_SCALE;
  x3_split8(x, part);
}

/* one tensor's block of rows: registers, then three planes of bf16 rows */
template <int DP>
struct Rows {
  static constexpr int R = block_rows(DP), P = pitch(DP), CPR = DP / 8;
  static constexpr int TASKS = (R * CPR + 255) / 256;
  f32x4 v[TASKS][2];
  TM_DEV void load(const float *base, int r0, int n, int D, int64_t ss, int tid) {
#pragma unroll
    for (int t = 0; t < TASKS; ++t) {
      const int i = tid + t * 256, row = r0 + i / CPR;
      load8(base + (int64_t)row * ss, (i % CPR) * 8, D, i < R * CPR && row < n, v[t]);
    }
  }
  TM_DEV void store(char *lds, int tid) const {
#pragma unroll
    for (int t = 0; t < TASKS; ++t) {
      const int i = tid + t * 256;
      if (R * CPR % 256 && i >= R * CPR) break;
      u32x4 part[3];
      split_run(v[t], part);
      const int at = tile_off<P>(i / CPR, i % CPR);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(u32x4 *)(lds + q * (R * P * 2) + at) = part[q];
    }
  }
};

/* this lane's row (query or key) as a split MFMA operand, per 32 columns */
template <int DP>
TM_DEV void own_row(const float *row, bool in, int D, int g, u32x4 (&part)[DP / 32][3]) {
#pragma unroll
  for (int ks = 0; ks < DP / 32; ++ks) {
    f32x4 v[2];
    load8(row, ks * 32 + 8 * g, D, in, v);
    split_run(v, part[ks]);
  }
}

/* 16 rows of a block (row r0 + c) as the row operand, 32 columns from 32 ks */
template <int DP>
TM_DEV void row_operand(uint32_t tile, uint32_t off, int r0, u32x4 (&part)[3]) {
  constexpr int P = pitch(DP), PLANE = block_rows(DP) * P * 2;
#pragma unroll
  for (int q = 0; q < 3; ++q) part[q] = lds_read16(tile + off + q * PLANE + r0 * P * 2);
}
/* 32 rows from r0 as the k-major operand, 16 columns */
template <int DP>
TM_DEV void k_operand(uint32_t tile, uint32_t off, int r0, u32x4 (&part)[3]) {
  constexpr int P = pitch(DP), PLANE = block_rows(DP) * P * 2;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    part[q] = lds_read_kmajor(tile + off, q * PLANE + r0 * P * 2, q * PLANE + (r0 + 16) * P * 2);
}
/* eight fp32 results of two 16-row tiles (rows 4g + r of each), `scale` times as
 * large, as the other operand of a k-major product */
TM_DEV void result_operand(const f32x4 &a, const f32x4 &b, float scale, u32x4 (&part)[3]) {
  float x[8] = {a[0] * scale, a[1] * scale, a[2] * scale, a[3] * scale,
                b[0] * scale, b[1] * scale, b[2] * scale, b[3] * scale};
  x3_split8(x, part);
}

/* what a product of two (three) split operands comes out as, undone */
constexpr float SCALE2 = X3_SCALE * X3_SCALE, UNSCALE2 = 1.f / SCALE2, UNSCALE3 = UNSCALE2 / X3_SCALE;
/* (a score scale below this would be rounded when UNSCALE2 is folded into it) */
TM_DEV bool scale_beyond(float qk_scale) { return fabsf(qk_scale) < 0x1p-90f; }
/* scores past the range, which the exponential would take to an ordinary 0: the
 * sum of 0 s is not 0 */
TM_DEV void note_finite(float &sum, float s) { sum = __builtin_fmaf(s, 0.f, sum); }

/* lane parts of the operand addresses */
template <int DP>
struct Lane {
  uint32_t row[DP / 32], km[DP / 16];
  TM_DEV Lane(int g, int c) {
#pragma unroll
    for (int ks = 0; ks < DP / 32; ++ks) row[ks] = (uint32_t)tile_off<pitch(DP)>(c, ks * 4 + g);
#pragma unroll
    for (int dt = 0; dt < DP / 16; ++dt)
      km[dt] = (uint32_t)(tile_off<pitch(DP)>(4 * g + (c >> 2), 2 * dt + ((c & 3) >> 1)) + ((c & 1) << 3));
  }
};

/* ---- forward: attn_fwd_generic's online softmax ------------------------------ */
template <int DP, bool CAUSAL>
TM_DEV void attn_fwd_x3(const TmAttnFwdArgs &p, char *lds) {
  constexpr int BM = 64, BN = block_rows(DP), KT = BN / 16, KS = DP / 32, DT = DP / 16;
  const uint32_t kb = lds_addr(lds), vb = kb + planes(DP);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.y, q0 = blockIdx.x * BM;
  const int n = p.n_ctx, D = p.head_dim;
  const int64_t base = (int64_t)bh * p.stride_head, ss = p.stride_seq;
  const float *Q = (const float *)p.q + base, *K = (const float *)p.k + base, *V = (const float *)p.v + base;
  const int qi = q0 + wave * 16 + c;
  u32x4 qf[KS][3];
  own_row<DP>(Q + (int64_t)qi * ss, qi < n, D, g, qf);
  const Lane<DP> at(g, c);
  const float qk_scale = p.sm_scale * TM_LOG2E, s_scale = qk_scale * UNSCALE2;
  float m_i = TM_NEG_INF, l_i = 0.f;
  f32x4 acc[DT], low[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = low[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int kend_all = CAUSAL ? min(n, q0 + BM) : n;
  const int nkb = (kend_all + BN - 1) / BN;
  const int split = blockIdx.z;
  const int kbeg = p.splits > 1 ? (int)((int64_t)split * nkb / p.splits) * BN : 0;
  const int kend = p.splits > 1 ? min(kend_all, (int)((int64_t)(split + 1) * nkb / p.splits) * BN) : kend_all;
  Rows<DP> kr, vr;
  if (kbeg < kend) {
    kr.load(K, kbeg, n, D, ss, tid);
    vr.load(V, kbeg, n, D, ss, tid);
  }
  float seen = 0.f;
  for (int k0 = kbeg; k0 < kend; k0 += BN) {
    __syncthreads();
    kr.store(lds, tid);
    vr.store(lds + planes(DP), tid);
    __syncthreads();
    if (k0 + BN < kend) {
      kr.load(K, k0 + BN, n, D, ss, tid);
      vr.load(V, k0 + BN, n, D, ss, tid);
    }
    f32x4 s[KT], sl[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) s[kt] = sl[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int kt = 0; kt < KT; kt += 2) {
        u32x4 a[2][3];
        row_operand<DP>(kb, at.row[ks], kt * 16, a[0]);
        row_operand<DP>(kb, at.row[ks], kt * 16 + 16, a[1]);
        mfma_x3<2>({&a[0], &a[1]}, {&qf[ks], &qf[ks]}, {&s[kt], &s[kt + 1]}, {&sl[kt], &sl[kt + 1]});
      }
    float mx = TM_NEG_INF;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int kj = k0 + kt * 16 + 4 * g + r;
        s[kt][r] += sl[kt][r];
        note_finite(seen, s[kt][r]);
        float v = s[kt][r] * s_scale;
        if (kj >= n || (CAUSAL && kj > qi)) v = TM_NEG_INF;
        s[kt][r] = v;
        mx = fmaxf(mx, v);
      }
    mx = group4_max(mx);
    const float m_new = fmaxf(m_i, mx);
    /* a row whose keys so far are all masked keeps P = 0 and l = 0 */
    const float m_use = m_new == TM_NEG_INF ? 0.f : m_new;
    float rs = 0.f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[kt][r] = exp2f(s[kt][r] - m_use);
        rs += s[kt][r];
      }
    const float alpha = exp2f(m_i - m_use);
    l_i = l_i * alpha + group4_sum(rs);
    m_i = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      acc[dt] *= alpha;
      low[dt] *= alpha;
    }
#pragma unroll
    for (int kk = 0; kk < BN / 32; ++kk) {
      u32x4 pf[3];
      result_operand(s[2 * kk], s[2 * kk + 1], X3_SCALE, pf);
#pragma unroll
      for (int dt = 0; dt < DT; dt += 2) {
        u32x4 a[2][3];
        k_operand<DP>(vb, at.km[dt], kk * 32, a[0]);
        k_operand<DP>(vb, at.km[dt + 1], kk * 32, a[1]);
        mfma_x3<2>({&a[0], &a[1]}, {&pf, &pf}, {&acc[dt], &acc[dt + 1]}, {&low[dt], &low[dt + 1]});
      }
    }
  }
  bool beyond = scale_beyond(qk_scale) || seen != 0.f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      acc[dt][r] += low[dt][r];
      beyond |= x3_not_finite(acc[dt][r]);
    }
  if (__syncthreads_or(beyond)) {
    attn_fwd_generic<float, DP, CAUSAL>(p, (float *)lds, (float *)lds + generic_tile(DP));
    return;
  }
  if (qi < n && p.splits > 1) {
    float *po = p.part + (((int64_t)split * p.heads + bh) * n + qi) * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = dt * 16 + 4 * g + r;
        if (d < D) po[d] = acc[dt][r] * UNSCALE2;
      }
    if (g == 0) {
      float *pml = p.part + (int64_t)p.splits * p.heads * n * D + (((int64_t)split * p.heads + bh) * n + qi) * 2;
      pml[0] = m_i;
      pml[1] = l_i;
    }
  } else if (qi < n) {
    float *O = (float *)p.o + base + (int64_t)qi * ss;
    const float inv = 1.f / l_i * UNSCALE2;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = dt * 16 + 4 * g + r;
        if (d < D) O[d] = acc[dt][r] * inv;
      }
    if (p.lse && g == 0) p.lse[(int64_t)bh * p.stride_lse + qi] = m_i + log2f(l_i);
  }
}

/* ---- dQ: attn_dq_generic's, 32 keys at a time ---------------------------------- */
template <int DP, bool CAUSAL>
TM_DEV void attn_dq_x3(const TmAttnDqArgs &p, char *lds) {
  constexpr int BM = 64, BN = block_rows(DP), KS = DP / 32, DT = DP / 16;
  /* the small products' accumulators live through the walk, or (past 64 columns,
   * where 256 registers do not hold them) through one block */
  constexpr bool KEEP = DP <= 64;
  const uint32_t kb = lds_addr(lds), vb = kb + planes(DP);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.y, q0 = blockIdx.x * BM;
  const int n = p.n_ctx, D = p.head_dim;
  const int64_t base = (int64_t)bh * p.stride_head, ss = p.stride_seq;
  const float *K = (const float *)p.k + base, *V = (const float *)p.v + base;
  const int qi = q0 + wave * 16 + c;
  u32x4 qf[KS][3], df[KS][3];
  own_row<DP>((const float *)p.q + base + (int64_t)qi * ss, qi < n, D, g, qf);
  own_row<DP>((const float *)p.dout + base + (int64_t)qi * ss, qi < n, D, g, df);
  const Lane<DP> at(g, c);
  const int64_t srow = (int64_t)bh * p.stride_lse + qi;
  const float lse = qi < n ? p.lse[srow] : 0.f;
  const float delta = qi < n ? p.delta[srow] * SCALE2 : 0.f; /* at dP's scale */
  const float qk_scale = p.sm_scale * TM_LOG2E, s_scale = qk_scale * UNSCALE2;
  float seen = 0.f;
  f32x4 acc[DT], low[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = low[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  /* ranges in 32-key blocks, as the generic kernel's: a range's first block may
   * start in the middle of one of BN */
  const int kend_all = CAUSAL ? min(n, q0 + BM) : n;
  const int nkb = (kend_all + 31) / 32;
  const int split = blockIdx.z;
  const int kbeg = p.splits > 1 ? (int)((int64_t)split * nkb / p.splits) * 32 : 0;
  const int kend = p.splits > 1 ? min(kend_all, (int)((int64_t)(split + 1) * nkb / p.splits) * 32) : kend_all;
  Rows<DP> kr, vr;
  if (kbeg < kend) {
    kr.load(K, kbeg, n, D, ss, tid);
    vr.load(V, kbeg, n, D, ss, tid);
  }
  for (int k0 = kbeg; k0 < kend; k0 += BN) {
    __syncthreads();
    kr.store(lds, tid);
    vr.store(lds + planes(DP), tid);
    __syncthreads();
    if (k0 + BN < kend) {
      kr.load(K, k0 + BN, n, D, ss, tid);
      vr.load(V, k0 + BN, n, D, ss, tid);
    }
#pragma unroll
    for (int kk = 0; kk < BN / 32; ++kk) {
      if (k0 + kk * 32 >= kend) break; /* the next range's */
      f32x4 s[2], dp[2], sl[2], dpl[2];
      s[0] = s[1] = dp[0] = dp[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
      sl[0] = sl[1] = dpl[0] = dpl[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          u32x4 a[2][3];
          row_operand<DP>(kb, at.row[ks], kk * 32 + t * 16, a[0]);
          row_operand<DP>(vb, at.row[ks], kk * 32 + t * 16, a[1]);
          mfma_x3<2>({&a[0], &a[1]}, {&qf[ks], &df[ks]}, {&s[t], &dp[t]}, {&sl[t], &dpl[t]});
          if (DP > 96) __builtin_amdgcn_sched_barrier(0); /* registers: the next reads not yet */
        }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int kj = k0 + kk * 32 + t * 16 + 4 * g + r;
          s[t][r] += sl[t][r];
          dp[t][r] += dpl[t][r];
          note_finite(seen, s[t][r]);
          float v = s[t][r] * s_scale;
          if (kj >= n || (CAUSAL && kj > qi)) v = TM_NEG_INF;
          s[t][r] = exp2f(v - lse) * (dp[t][r] - delta);
        }
      u32x4 dsf[3];
      result_operand(s[0], s[1], 1.f, dsf);
#pragma unroll
      for (int dt = 0; dt < DT; dt += 2) {
        u32x4 a[2][3];
        k_operand<DP>(kb, at.km[dt], kk * 32, a[0]);
        k_operand<DP>(kb, at.km[dt + 1], kk * 32, a[1]);
        if constexpr (KEEP) {
          mfma_x3<2>({&a[0], &a[1]}, {&dsf, &dsf}, {&acc[dt], &acc[dt + 1]}, {&low[dt], &low[dt + 1]});
        } else {
          f32x4 l[2] = {};
          mfma_x3<2>({&a[0], &a[1]}, {&dsf, &dsf}, {&acc[dt], &acc[dt + 1]}, {&l[0], &l[1]});
          acc[dt] += l[0];
          acc[dt + 1] += l[1];
        }
      }
    }
  }
  bool beyond = scale_beyond(qk_scale) || seen != 0.f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      acc[dt][r] += low[dt][r];
      beyond |= x3_not_finite(acc[dt][r]);
    }
  if (__syncthreads_or(beyond)) {
    attn_dq_generic<float, DP, CAUSAL>(p, (float *)lds, (float *)lds + generic_tile(DP));
    return;
  }
  if (qi < n) {
    float *po = p.splits > 1 ? p.part + (((int64_t)split * p.heads + bh) * n + qi) * D : nullptr;
    float *dq = (float *)p.dq + base + (int64_t)qi * ss;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = dt * 16 + 4 * g + r;
        if (d >= D) continue;
        const float x = acc[dt][r] * UNSCALE3;
        if (po) po[d] = x;
        else dq[d] = x * p.sm_scale;
      }
  }
}

/* ---- dK, dV: attn_dkdv_generic's, 32 queries at a time -------------------------- */
template <int DP, bool CAUSAL>
TM_DEV void attn_dkdv_x3(const TmAttnDkdvArgs &p, char *lds, float *Ls, float *Ds) {
  constexpr int BN = 64, BM = block_rows(DP), KS = DP / 32, DT = DP / 16;
  /* one wave per SIMD (past 64 columns) has only its own MFMAs to wait beside */
  constexpr bool WIDE = DP > 64;
  const uint32_t qb = lds_addr(lds), ob = qb + planes(DP);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int bh = blockIdx.y, k0 = blockIdx.x * BN;
  const int n = p.n_ctx, D = p.head_dim;
  const int64_t base = (int64_t)bh * p.stride_head, ss = p.stride_seq;
  const float *Q = (const float *)p.q + base, *dO = (const float *)p.dout + base;
  const float *Lrow = p.lse + (int64_t)bh * p.stride_lse, *Drow = p.delta + (int64_t)bh * p.stride_lse;
  const int kj = k0 + wave * 16 + c;
  u32x4 kf[KS][3], vf[KS][3];
  own_row<DP>((const float *)p.k + base + (int64_t)kj * ss, kj < n, D, g, kf);
  own_row<DP>((const float *)p.v + base + (int64_t)kj * ss, kj < n, D, g, vf);
  const Lane<DP> at(g, c);
  const float qk_scale = p.sm_scale * TM_LOG2E, s_scale = qk_scale * UNSCALE2;
  float seen = 0.f;
  f32x4 dk[DT], dv[DT], dkl[DT], dvl[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dk[dt] = dv[dt] = dkl[dt] = dvl[dt] = (f32x4){0.f, 0.f, 0.f, 0.f};

  /* ranges in 32-query blocks, as the generic kernel's */
  const int qfirst = CAUSAL ? k0 : 0;
  const int nqb = (n - qfirst + 31) / 32;
  const int split = blockIdx.z;
  const int qstart = p.splits > 1 ? qfirst + (int)((int64_t)split * nqb / p.splits) * 32 : qfirst;
  const int qstop = p.splits > 1 ? min(n, qfirst + (int)((int64_t)(split + 1) * nqb / p.splits) * 32) : n;
  Rows<DP> qr, dor;
  float l_next = 0.f, d_next = 0.f; /* thread tid < BM: L and Delta of row tid */
  auto load = [&](int q0) {
    qr.load(Q, q0, n, D, ss, tid);
    dor.load(dO, q0, n, D, ss, tid);
    const int qi = q0 + tid;
    l_next = tid < BM && qi < n ? Lrow[qi] : 0.f;
    d_next = tid < BM && qi < n ? Drow[qi] * SCALE2 : 0.f; /* at dP's scale */
  };
  if (qstart < qstop) load(qstart);
  for (int q0 = qstart; q0 < qstop; q0 += BM) {
    __syncthreads();
    qr.store(lds, tid);
    dor.store(lds + planes(DP), tid);
    if (tid < BM) {
      Ls[tid] = l_next;
      Ds[tid] = d_next;
    }
    __syncthreads();
    if (q0 + BM < qstop) load(q0 + BM);
#pragma unroll
    for (int kk = 0; kk < BM / 32; ++kk) {
      if (q0 + kk * 32 >= qstop) break; /* the next range's */
      f32x4 s[2], dp[2], sl[2], dpl[2];
      s[0] = s[1] = dp[0] = dp[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
      sl[0] = sl[1] = dpl[0] = dpl[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < (WIDE ? KS : 2 * KS); ++i) {
        const int ks = WIDE ? i : i % KS, t = i / KS;
        u32x4 a[2][3], b[2][3];
        row_operand<DP>(qb, at.row[ks], kk * 32 + t * 16, a[0]);
        row_operand<DP>(ob, at.row[ks], kk * 32 + t * 16, a[1]);
        if constexpr (WIDE) {
          row_operand<DP>(qb, at.row[ks], kk * 32 + 16, b[0]);
          row_operand<DP>(ob, at.row[ks], kk * 32 + 16, b[1]);
          mfma_x3<4>({&a[0], &a[1], &b[0], &b[1]}, {&kf[ks], &vf[ks], &kf[ks], &vf[ks]},
                     {&s[0], &dp[0], &s[1], &dp[1]}, {&sl[0], &dpl[0], &sl[1], &dpl[1]});
        } else {
          mfma_x3<2>({&a[0], &a[1]}, {&kf[ks], &vf[ks]}, {&s[t], &dp[t]}, {&sl[t], &dpl[t]});
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = kk * 32 + t * 16 + 4 * g + r, qi = q0 + row;
          s[t][r] += sl[t][r];
          dp[t][r] += dpl[t][r];
          note_finite(seen, s[t][r]);
          float v = s[t][r] * s_scale;
          if (qi >= n || (CAUSAL && qi < kj)) v = TM_NEG_INF;
          s[t][r] = exp2f(v - Ls[row]);
          dp[t][r] = s[t][r] * (dp[t][r] - Ds[row]);
        }
      u32x4 pf[3], dsf[3];
      result_operand(s[0], s[1], X3_SCALE, pf);
      result_operand(dp[0], dp[1], 1.f, dsf);
#pragma unroll
      for (int dt = 0; dt < DT; dt += WIDE ? 2 : 1) {
        u32x4 a[2][3], b[2][3];
        k_operand<DP>(ob, at.km[dt], kk * 32, a[0]);
        k_operand<DP>(qb, at.km[dt], kk * 32, a[1]);
        if constexpr (WIDE) {
          k_operand<DP>(ob, at.km[dt + 1], kk * 32, b[0]);
          k_operand<DP>(qb, at.km[dt + 1], kk * 32, b[1]);
          mfma_x3<4>({&a[0], &a[1], &b[0], &b[1]}, {&pf, &dsf, &pf, &dsf},
                     {&dv[dt], &dk[dt], &dv[dt + 1], &dk[dt + 1]}, {&dvl[dt], &dkl[dt], &dvl[dt + 1], &dkl[dt + 1]});
        } else {
          mfma_x3<2>({&a[0], &a[1]}, {&pf, &dsf}, {&dv[dt], &dk[dt]}, {&dvl[dt], &dkl[dt]});
        }
      }
    }
  }
  bool beyond = scale_beyond(qk_scale) || seen != 0.f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dk[dt][r] += dkl[dt][r];
      dv[dt][r] += dvl[dt][r];
      beyond |= kj < n && (x3_not_finite(dk[dt][r]) || x3_not_finite(dv[dt][r]));
    }
  if (__syncthreads_or(beyond)) {
    attn_dkdv_generic<float, DP, CAUSAL>(p, (float *)lds, (float *)lds + generic_tile(DP), Ls, Ds);
    return;
  }
  if (kj < n) {
    const int64_t plane = (int64_t)p.heads * n * D;
    float *pk = p.splits > 1 ? p.part + 2 * split * plane + ((int64_t)bh * n + kj) * D : nullptr;
    float *dK = (float *)p.dk + base + (int64_t)kj * ss, *dV = (float *)p.dv + base + (int64_t)kj * ss;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = dt * 16 + 4 * g + r;
        if (d >= D) continue;
        const float k = dk[dt][r] * UNSCALE3, v = dv[dt][r] * UNSCALE2;
        if (pk) {
          pk[d] = k;
          pk[plane + d] = v;
        } else {
          dK[d] = k * p.sm_scale;
          dV[d] = v;
        }
      }
  }
}

} // namespace

#define TM_ATTN_X3(DP, CAUSAL, CN)                                                            \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void   \
  tm_attn_fwd_generic_f32_d##DP##CN(TmAttnFwdArgs p) {                                        \
    __shared__ __align__(1024) char lds[lds_bytes(DP)];                                       \
    attn_fwd_x3<DP, CAUSAL>(p, lds);                                                          \
  }                                                                                           \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void   \
  tm_attn_dq_generic_f32_d##DP##CN(TmAttnDqArgs p) {                                          \
    __shared__ __align__(1024) char lds[lds_bytes(DP)];                                       \
    attn_dq_x3<DP, CAUSAL>(p, lds);                                                           \
  }                                                                                           \
  /* (K and V in registers beside both accumulators: past 64 columns 256 registers \
   * spill) */                                                                                \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DP <= 64 ? 2 : 1))) void \
  tm_attn_dkdv_generic_f32_d##DP##CN(TmAttnDkdvArgs p) {                                      \
    __shared__ __align__(1024) char lds[lds_bytes(DP)];                                       \
    __shared__ float l[64], dl[64];                                                           \
    attn_dkdv_x3<DP, CAUSAL>(p, lds, l, dl);                                                  \
  }
#define TM_ATTN_X3_DP(DP)     \
  TM_ATTN_X3(DP, false, )     \
  TM_ATTN_X3(DP, true, _causal)
TM_ATTN_X3_DP(32)
TM_ATTN_X3_DP(64)
TM_ATTN_X3_DP(96)
TM_ATTN_X3_DP(128)
