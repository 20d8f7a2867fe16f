/*
 * gfx950 GEMM for fp32 on the bf16 matrix cores: every operand is split into
 * three bf16 parts (split3.h), and C = A @ B is eight of their nine products, hi hi
 * in one fp32 accumulator and the seven small ones in another.  A 16x16x32 bf16
 * MFMA rounds once per 32 products where the 16x16x4 fp32 one rounds per 4, so
 * dense results are closer to the exact ones than the fp32 MFMA's (relative error
 * at K = 64, 1025 and 4097: 1.4, 5.7 and 11.4e-7 on that, 0.5, 0.9 and 1.2e-7
 * here) and a lone product is as close (0.51 of its last place at most, 0.50 on
 * the fp32 MFMA).  Six products in one accumulator took 15% less time and were up
 * to 1.41 off there.  Eight bf16 MFMAs take half the fp32 MFMA's time.
 *
 * Measured (us, fp32 MFMA kernels before and now): 2049 x 3079 x 1025 177 and
 * 111, 4096^3 1050 and 754 (182 TFLOP/s), 1500^3 121 and 75, 1000^3 43 and 31, 129 x
 * 202 x 7481 273 and 29.  The MFMA pipes are busy 64% of the time at 4096^3, at the
 * power limit's clock, and 42% at 2049 x 3079 x 1025, whose 425 tiles fill 0.83 of a
 * round; the rest is what two workgroups per CU leave uncovered of the split (6 VALU
 * operations an element), the LDS writes and transposed reads between its barriers.
 * Splitting into registers behind the MFMAs instead ran 93 / 738 us, three
 * workgroups per CU (168 registers) 114 / 818.
 *
 * What the split cannot represent goes back to fp32: values and results near the
 * top of the range (split3.h), infinities and NaN leave a non-finite accumulator; a
 * workgroup that meets one computes its tile again on v_mfma_f32_16x16x4_f32.
 */
#include "gemm_fast.h"
#include "split3.h"
#include "x3_runs.h"

namespace {

constexpr int XK = 32; /* k per step */

typedef f32x4 f32x4_any __attribute__((aligned(4)));

/* A [TILE rows][32 k] plane (k contiguous): 64-byte rows of four 16-byte chunks,
 * chunk c of row r at c ^ ((r >> 2) & 3): 16 rows at one chunk (ds_read_b128 of
 * an operand) then cover the 256-byte bank row. */
TM_DEV int x3_off(int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 2) & 3)) << 4); }

/* One operand's tile: TILE x 32 floats through registers, eight per task, into
 * three bf16 planes of TILE * 64 bytes.  CONTIG: k is the contiguous dimension
 * (planes [TILE][32]), else the other one is (planes [32][TILE], gemm_fast.h's
 * B layout).  Loads are 16 bytes at any 4-byte address, where x3_runs.h says.
 * What is then not of the matrix is replaced by zeros: k past K because it would
 * be added, columns so that a stray value does not send the workgroup to its fp32
 * path. */
template <bool CONTIG, int TILE>
struct X3Tile {
  static constexpr int TASKS = TILE / 64, CPR = CONTIG ? 4 : TILE / 8, RPT = 256 / CPR;
  static constexpr int PLANE = TILE * XK * 2;
  /* bytes from the tile's first element; k-major tasks lie RPT rows apart */
  uint32_t off[CONTIG ? TASKS : 1][2];
  f32x4 v[TASKS][2];
  int row0, chunk, width;

  TM_DEV void init(int64_t ld, int rows, int tid) { /* rows: of the matrix, from the tile's first */
    width = CONTIG ? TILE : rows;
    row0 = tid / CPR;
    chunk = tid % CPR;
#pragma unroll
    for (int t = 0; t < TASKS; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        off[t][h] = x3_run<CONTIG>(ld, row0 + t * RPT, chunk * 8 + h * 4, rows);
      }
  }
  TM_DEV void load(const float *base, int64_t ld, int k_left) {
    const char *src = (const char *)base;
    if (k_left >= XK) {
#pragma unroll
      for (int t = 0; t < TASKS; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[t][h] = *(const f32x4_any *)(CONTIG ? src + off[t][h] : src + 4 * t * RPT * ld + off[0][h]);
    } else {
#pragma unroll
      for (int t = 0; t < TASKS; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int row = row0 + t * RPT, col = chunk * 8 + h * 4;
          const uint32_t run = CONTIG ? off[t][h] : off[0][h] + 4 * (uint32_t)(t * RPT * ld);
          const f32x4 x = *(const f32x4_any *)(src + x3_last_run<CONTIG>(run, ld, row, col, k_left));
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t][h][e] = (CONTIG ? col + e : row) < k_left ? x[e] : 0.f;
        }
    }
    if (!CONTIG && width < TILE) {
#pragma unroll
      for (int t = 0; t < TASKS; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (chunk * 8 + h * 4 + e >= width) v[t][h][e] = 0.f;
    }
  }
  /* split into the planes at `lds` */
  TM_DEV void store(char *lds) {
#pragma unroll
    for (int t = 0; t < TASKS; ++t) {
      const int row = row0 + t * RPT;
      const int at = CONTIG ? x3_off(row, chunk) : b_off<TILE>(row, chunk);
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = v[t][e >> 2][e & 3] * X3_SCALE;
      u32x4 part[3];
      x3_split8(x, part);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(u32x4 *)(lds + q * PLANE + at) = part[q];
    }
  }
  /* unsplit, for the fp32 MFMAs: rows of 36 floats (CONTIG), or of TILE + 16, where
   * the 64 lanes of a read (16 rows or columns at four k) fall on 64 banks */
  static constexpr int F32_LD = CONTIG ? XK + 4 : TILE + 16;
  static_assert((CONTIG ? TILE : XK) * F32_LD * 4 <= 3 * PLANE, "LDS");
  TM_DEV void store_f32(char *lds) {
#pragma unroll
    for (int t = 0; t < TASKS; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *(f32x4 *)(lds + ((row0 + t * RPT) * F32_LD + chunk * 8 + h * 4) * 4) = v[t][h];
  }
  TM_DEV float read_f32(const char *lds, int row, int k) {
    return ((const float *)lds)[CONTIG ? row * F32_LD + k : k * F32_LD + row];
  }
};

/* One 256-thread workgroup (4 waves, 2 x 2) per TILE x TILE tile of C; grid y
 * and p.splits give it a range of the k-steps, whose fp32 partial then goes to
 * p.part.  A step's tiles are loaded into registers while the previous step's
 * MFMAs run, and split into one set of LDS planes between two barriers; two or
 * three workgroups to a CU fill each other's gaps. */
template <int EPI, int TILE, bool BT, bool AT>
TM_DEV void gemm_x3(const TmGemmArgs &p) {
  constexpr int WT = TILE / 2, NI = WT / 16;
  constexpr int PLANE = TILE * XK * 2;
  __shared__ __align__(1024) char lds_a[3 * PLANE];
  __shared__ __align__(1024) char lds_b[3 * PLANE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;

  const int mt = (p.m + TILE - 1) / TILE, nt = (p.n + TILE - 1) / TILE;
  const int logical = g_xcd_remap(blockIdx.x, gridDim.x);
  constexpr int GROUP = 8;
  const int per_group = GROUP * nt;
  const int group = logical / per_group;
  const int first_m = group * GROUP;
  const int gm = min(mt - first_m, GROUP);
  const int in_group = logical - group * per_group;
  const int m0 = (first_m + in_group % gm) * TILE, n0 = (in_group / gm) * TILE;

  const int64_t lda = AT ? p.sak : p.sam, ldb = BT ? p.sbn : p.sbk;
  const float *A = (const float *)p.a + (AT ? (int64_t)m0 : (int64_t)m0 * lda);
  const float *B = (const float *)p.b + (BT ? (int64_t)n0 * ldb : (int64_t)n0);
  const int rows = min(p.m - m0, TILE), cols = min(p.n - n0, TILE);

  const int ksteps = (p.k + XK - 1) / XK;
  const int splits = p.splits > 1 ? p.splits : 1;
  const int split = splits > 1 ? (int)blockIdx.y : 0;
  const int kbeg = (int)((int64_t)split * ksteps / splits);
  const int kend = (int)((int64_t)(split + 1) * ksteps / splits);

  X3Tile<!AT, TILE> ta;
  X3Tile<BT, TILE> tb;
  ta.init(lda, rows, tid);
  tb.init(ldb, cols, tid);
  auto load = [&](int kb) {
    const int k0 = kb * XK;
    ta.load(AT ? A + (int64_t)k0 * lda : A + k0, lda, p.k - k0);
    tb.load(BT ? B + k0 : B + (int64_t)k0 * ldb, ldb, p.k - k0);
  };
  f32x4 acc[NI][NI], low[NI][NI]; /* the hi hi products, the small ones */
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = low[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  if (kbeg < kend) load(kbeg);
  for (int kb = kbeg; kb < kend; ++kb) {
    ta.store(lds_a);
    tb.store(lds_b);
    __syncthreads();
    if (kb + 1 < kend) load(kb + 1);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 bf[3][NI];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int n = wn * WT + j * 16;
        const u32x4 x = BT ? *(const u32x4 *)(lds_b + q * PLANE + x3_off(n + c, g))
                           : read_b_operand<TILE>(lds_b + q * PLANE, 0, n, g, c);
        bf[q][j] = __builtin_bit_cast(bf16x8, x);
      }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      bf16x8 af[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int m = wm * WT + i * 16;
        const u32x4 x = AT ? read_b_operand<TILE>(lds_a + q * PLANE, 0, m, g, c)
                           : *(const u32x4 *)(lds_a + q * PLANE + x3_off(m + c, g));
        af[q] = __builtin_bit_cast(bf16x8, x);
      }
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = mfma_16x16x32(bf[0][j], af[0], acc[i][j]);
#pragma unroll
      for (int order = 1; order <= 3; ++order)
#pragma unroll
        for (int q = order < 3 ? 0 : 1; q <= order && q < 3; ++q)
#pragma unroll
          for (int j = 0; j < NI; ++j) low[i][j] = mfma_16x16x32(bf[q][j], af[order - q], low[i][j]);
    }
    __syncthreads();
  }

  bool beyond = false;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        acc[i][j][r] += low[i][j][r];
        beyond |= x3_not_finite(acc[i][j][r]);
        acc[i][j][r] *= 1.f / (X3_SCALE * X3_SCALE);
      }
  if (__syncthreads_or(beyond)) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (kbeg < kend) load(kbeg);
    for (int kb = kbeg; kb < kend; ++kb) {
      ta.store_f32(lds_a);
      tb.store_f32(lds_b);
      __syncthreads();
      if (kb + 1 < kend) load(kb + 1);
#pragma unroll
      for (int k = 0; k < XK; k += 4) {
        float a[NI], b[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          a[i] = ta.read_f32(lds_a, wm * WT + i * 16 + c, k + g);
          b[i] = tb.read_f32(lds_b, wn * WT + i * 16 + c, k + g);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = mfma_f32_16x16x4(b[j], a[i], acc[i][j]);
      }
      __syncthreads();
    }
  }

  /* acc[i][j] is the C^T tile: lane holds row m0 + wm*WT + i*16 + c, columns
   * n0 + wn*WT + j*16 + 4g .. +3 */
  if (splits > 1) {
    const int64_t np = (p.n + 3) & ~3;
    float *part = p.part + (int64_t)split * p.m * np;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int m = m0 + wm * WT + i * 16 + c, n = n0 + wn * WT + j * 16 + 4 * g;
        if (m < p.m && n < p.n) *(f32x4 *)(part + m * np + n) = acc[i][j];
      }
    return;
  }
  f32x4 bias[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + wn * WT + j * 16 + 4 * g + r;
      bias[j][r] = EPI == EPI_BIAS_RELU && n < p.n ? ((const float *)p.bias)[n] : 0.f;
    }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int m = m0 + wm * WT + i * 16 + c;
    if (m >= p.m) continue;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n0 + wn * WT + j * 16 + 4 * g;
      f32x4 v = acc[i][j];
      if (EPI == EPI_BIAS_RELU) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r] + bias[j][r], 0.f);
      }
      float *dst = (float *)p.c + (int64_t)m * p.scm + n;
      if (n + 4 <= p.n) {
        *(f32x4_any *)dst = v;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.n) dst[r] = v[r];
      }
    }
  }
}

/* The ranges' partials summed in order into C, with the epilogue */
template <int EPI>
TM_DEV void gemm_x3_reduce(const TmGemmArgs &p) {
  const int64_t np4 = (p.n + 3) >> 2;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)p.m * np4) return;
  const int64_t m = idx / np4;
  const int n = (int)(idx - m * np4) * 4;
  const int64_t plane = (int64_t)p.m * np4 * 4;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < p.splits; ++s) sum += *(const f32x4 *)(p.part + s * plane + m * np4 * 4 + n);
  float *dst = (float *)p.c + m * p.scm + n;
  for (int r = 0; r < 4 && n + r < p.n; ++r)
    dst[r] = EPI == EPI_BIAS_RELU ? fmaxf(sum[r] + ((const float *)p.bias)[n + r], 0.f) : sum[r];
}

} // namespace

#define TM_X3(NAME, EPI, TILE, BT, AT)                                                        \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void   \
  NAME(TmGemmArgs p) {                                                                        \
    gemm_x3<EPI, TILE, BT, AT>(p);                                                            \
  }
TM_X3(tm_gemm_x3_f32, EPI_NONE, 128, false, false)
TM_X3(tm_gemm_x3_nt_f32, EPI_NONE, 128, true, false)
TM_X3(tm_gemm_x3_tn_f32, EPI_NONE, 128, false, true)
TM_X3(tm_sae_x3_f32, EPI_BIAS_RELU, 128, false, false)
TM_X3(tm_gemm_x3_t64_f32, EPI_NONE, 64, false, false)
TM_X3(tm_gemm_x3_nt_t64_f32, EPI_NONE, 64, true, false)
TM_X3(tm_gemm_x3_tn_t64_f32, EPI_NONE, 64, false, true)
TM_X3(tm_sae_x3_t64_f32, EPI_BIAS_RELU, 64, false, false)
extern "C" __global__ __launch_bounds__(256) void tm_gemm_split_reduce_f32(TmGemmArgs p) {
  gemm_x3_reduce<EPI_NONE>(p);
}
extern "C" __global__ __launch_bounds__(256) void tm_sae_split_reduce_f32(TmGemmArgs p) {
  gemm_x3_reduce<EPI_BIAS_RELU>(p);
}
