#ifndef TM_GEMM_GENERIC_H
#define TM_GEMM_GENERIC_H

#include "common.h"

/* ---------------------------------------------------------------------------
 * matmul_kernel: C = A @ B, masked in M, N and K, f32 accumulation, output in
 * the element type (GEMMKernel.swift:28-174; matmul.py:20-44).
 * 64x64 output tile per 256-thread workgroup, 4 waves in 2x2, 32x32 per wave.
 * K advances 32 at a time; the next k-slice's global loads are issued into
 * registers before the current slice's MFMAs, so their latency overlaps the
 * contraction (one barrier-separated LDS store per slice).
 * ------------------------------------------------------------------------- */
constexpr int GENERIC_A = 64 * 33, GENERIC_B = 32 * 68; /* floats of its two LDS tiles */
template <typename T, int EPI>
TM_DEV void gemm_generic(const TmGemmArgs &p, float *a_lds, float *b_lds) {
  constexpr int BM = 64, BN = 64, BK = 32;
  constexpr int PER = BM * BK / 256; /* elements of A (and of B) per thread per slice */
  float(*As)[BK + 1] = (float(*)[BK + 1])a_lds;
  float(*Bs)[BN + 4] = (float(*)[BN + 4])b_lds;
  const T *A = (const T *)p.a;
  const T *B = (const T *)p.b;
  T *C = (T *)p.c;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;

  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  /* element e = tid + 256 * i of a slice: A row e / BK, column e % BK (k
   * fastest, so a wave reads runs along A's rows); B row e / BN, column e % BN */
  float ra[PER], rb[PER];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 256 * i;
      const int gm = m0 + e / BK, gk = k0 + e % BK;
      ra[i] = (gm < p.m && gk < p.k) ? to_f32(A[(int64_t)gm * p.sam + (int64_t)gk * p.sak]) : 0.f;
      const int kk = k0 + e / BN, gn = n0 + e % BN;
      rb[i] = (kk < p.k && gn < p.n) ? to_f32(B[(int64_t)kk * p.sbk + (int64_t)gn * p.sbn]) : 0.f;
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = tid + 256 * i;
      As[e / BK][e % BK] = ra[i];
      Bs[e / BN][e % BN] = rb[i];
    }
  };

  if (p.k > 0) load(0);
  for (int k0 = 0; k0 < p.k; k0 += BK) {
    store();
    __syncthreads();
    if (k0 + BK < p.k) load(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = As[wm * 32 + i * 16 + c][kk + g];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = Bs[kk + g][wn * 32 + j * 16 + c];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f32_16x16x4(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }

  /* the bias of this lane's two columns, loaded before any store to C */
  float bias[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = n0 + wn * 32 + j * 16 + c;
    bias[j] = (EPI == EPI_BIAS_RELU && col < p.n) ? to_f32(((const T *)p.bias)[col]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + wm * 32 + i * 16 + 4 * g + r;
        const int col = n0 + wn * 32 + j * 16 + c;
        const float v = EPI == EPI_BIAS_RELU ? fmaxf(acc[i][j][r] + bias[j], 0.f) : acc[i][j][r];
        if (row < p.m && col < p.n) C[(int64_t)row * p.scm + (int64_t)col * p.scn] = from_f32<T>(v);
      }
}

#endif
