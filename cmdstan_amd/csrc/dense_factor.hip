// Cholesky factor and its inverse for every chain's given dense metric (the
// metric a run starts from), a block of eight waves per chain, on FP64 matrix
// cores.  A = L L^T, column-major: L on and below the diagonal of the output,
// row r of X = L^-1 in column r above it (dense_tri_sample reads both).
//
// Panels of 32 columns.  Left-looking: the panel's update A - L L_J^T is a
// product over the columns done so far, both operands read straight from
// global memory (lanes of a quarter wave take 16 consecutive rows of one
// column: 128-byte segments, no LDS).  One wave factors the 32 x 32 diagonal
// block and inverts it with rows and columns in registers; the rows below are
// one more product with that inverse.  Then block rows of X: X_R = -X_RR (L_R X)
// from the block rows above.
//
// Bound: the chain of D / 32 panels, each a factorisation of its diagonal
// block (some 12 thousand dependent cycles) and two products of little depth.
// Before, one wave walked D columns with a pivot sum each and the inverse row by
// row: 144 ms for 64 chains at D = 520 (two dependent passes over L per column);
// now 2.1 ms.
#include "device_common.h"
#include "launch.h"

namespace nutsgpu {

typedef double d4 __attribute__((ext_vector_type(4)));
#define DF_NB 32
#define DF_W 8

__device__ __forceinline__ void df_sync() {  // the block's global writes visible to all its waves
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __syncthreads();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ double df_lane(double v, int j) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), j),
                          __builtin_amdgcn_readlane(__double2loint(v), j));
}

__global__ void __launch_bounds__(64 * DF_W, 2) dense_factor_kernel(NutsBuffers B, int* __restrict__ failed) {
  __shared__ double sD[DF_NB][DF_NB + 1], sT[DF_NB][DF_NB + 1];
  __shared__ double sS[DF_W][DF_NB][17];
  __shared__ int bad;
  const int c = blockIdx.x;
  const int D = B.D[c];
  const double* A = B.dM + B.moff[c];
  double* L = B.dL + B.moff[c];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, lr = l & 15, lk = l >> 4;
  const int last = D - 1;
  if (tid == 0) bad = 0;
  __syncthreads();

  for (int j0 = 0; j0 < D; j0 += DF_NB) {
    const int nb = min(DF_NB, D - j0);
    // panel columns j0 + m (result rows), matrix rows i0 + n (result columns)
    const int m0 = min(j0 + lr, last), m1 = min(j0 + 16 + lr, last);
    for (int i0 = j0 + 16 * w; i0 < D; i0 += 16 * DF_W) {
      const int n = min(i0 + lr, last);
      d4 a0 = d4{0, 0, 0, 0}, a1 = d4{0, 0, 0, 0};
#pragma unroll 4
      for (int k = 0; k < j0; k += 4) {
        const double* col = L + (int64_t)(k + lk) * D;
        const double x = col[n], p0 = col[m0], p1 = col[m1];
        a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x, a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x, a1, 0, 0, 0);
      }
      const int row = i0 + lr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = j0 + 4 * i + lk;
        if (row < D && m < D && row >= m) L[(int64_t)m * D + row] = A[(int64_t)m * D + row] - a0[i];
        if (row < D && m + 16 < D && row >= m + 16)
          L[(int64_t)(m + 16) * D + row] = A[(int64_t)(m + 16) * D + row] - a1[i];
      }
    }
    df_sync();
    if (w == 0) {
      // lane r (< 32) holds row r of the diagonal block, padded to 32 with a unit block
      const int r = l & 31;
      double v[DF_NB];
#pragma unroll
      for (int q = 0; q < DF_NB; ++q)
        v[q] = r < nb && q < nb ? (q <= r ? L[(int64_t)(j0 + q) * D + j0 + r] : 0.0) : (q == r ? 1.0 : 0.0);
      bool pd = true;
#pragma unroll
      for (int q = 0; q < DF_NB; ++q) {
        const double piv = df_lane(v[q], q);
        pd = pd && piv > 0;
        const double d = sqrt(piv);
        v[q] = r == q ? d : v[q] / d;
#pragma unroll
        for (int s = q + 1; s < DF_NB; ++s) v[s] -= v[q] * df_lane(v[q], s);
      }
      if (l == 0 && !pd) bad = 1;
      if (l < DF_NB) {
#pragma unroll
        for (int q = 0; q < DF_NB; ++q) sD[r][q] = q <= r ? v[q] : 0.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // lane c holds column c of the inverse
      double x[DF_NB];
#pragma unroll
      for (int q = 0; q < DF_NB; ++q) {
        double s = q == r ? 1.0 : 0.0;
#pragma unroll
        for (int k = 0; k < q; ++k) s -= sD[q][k] * x[k];
        x[q] = q < r ? 0.0 : s / sD[q][q];
      }
      if (l < DF_NB) {
#pragma unroll
        for (int q = 0; q < DF_NB; ++q) sT[q][r] = x[q];
      }
    }
    __syncthreads();
    if (bad) {
      if (tid == 0) atomicAdd(failed, 1);
      return;
    }
    // the diagonal block: L below, its inverse's rows above (row r in column r)
    for (int e = tid; e < nb * nb; e += 64 * DF_W) {
      const int q = e / nb, r = e % nb;  // column j0 + q, row j0 + r
      L[(int64_t)(j0 + q) * D + j0 + r] = r >= q ? sD[r][q] : sT[q][r];
    }
    // rows below: L(i, J) = P(i, J) T^T
    for (int i0 = j0 + DF_NB + 16 * w; i0 < D; i0 += 16 * DF_W) {
      const int n = min(i0 + lr, last);
      double p[DF_NB / 4];
#pragma unroll
      for (int s = 0; s < DF_NB / 4; ++s) p[s] = L[(int64_t)(j0 + 4 * s + lk) * D + n];
      d4 a0 = d4{0, 0, 0, 0}, a1 = d4{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < DF_NB / 4; ++s) {
        if (s < 4) a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(sT[lr][4 * s + lk], p[s], a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(sT[16 + lr][4 * s + lk], p[s], a1, 0, 0, 0);
      }
      if (i0 + lr < D) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          L[(int64_t)(j0 + 4 * i + lk) * D + i0 + lr] = a0[i];
          L[(int64_t)(j0 + 16 + 4 * i + lk) * D + i0 + lr] = a1[i];
        }
      }
    }
    df_sync();
  }

  for (int r0 = DF_NB; r0 < D; r0 += DF_NB) {
    for (int e = tid; e < DF_NB * DF_NB; e += 64 * DF_W) {
      const int r = e / DF_NB, q = e % DF_NB;  // T[r][q] of the diagonal block's inverse
      const int rr = r0 + r, qq = r0 + q;
      sT[r][q] = rr < D && q <= r ? (q == r ? 1.0 / L[(int64_t)rr * D + rr] : L[(int64_t)rr * D + qq]) : 0.0;
    }
    __syncthreads();
    const int m0 = min(r0 + lr, last), m1 = min(r0 + 16 + lr, last);
    for (int c0 = 16 * w; c0 < r0; c0 += 16 * DF_W) {
      const int n = c0 + lr;
      d4 a0 = d4{0, 0, 0, 0}, a1 = d4{0, 0, 0, 0};
      // rows k of X start at its diagonal: the first 16 are masked
#pragma unroll
      for (int k = c0; k < c0 + 16; k += 4) {
        const double* col = L + (int64_t)(k + lk) * D;
        const double u = col[n];  // n <= k: X[k][n] or, at n == k, L[k][k]
        const double x = n < k + lk ? u : (n == k + lk ? 1.0 / u : 0.0);
        a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(col[m0], x, a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(col[m1], x, a1, 0, 0, 0);
      }
#pragma unroll 4
      for (int k = c0 + 16; k < r0; k += 4) {
        const double* col = L + (int64_t)(k + lk) * D;
        const double x = col[n], p0 = col[m0], p1 = col[m1];
        a0 = __builtin_amdgcn_mfma_f64_16x16x4f64(p0, x, a0, 0, 0, 0);
        a1 = __builtin_amdgcn_mfma_f64_16x16x4f64(p1, x, a1, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sS[w][4 * i + lk][lr] = a0[i];
        sS[w][16 + 4 * i + lk][lr] = a1[i];
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      d4 y0 = d4{0, 0, 0, 0}, y1 = d4{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < DF_NB / 4; ++s) {
        const double x = sS[w][4 * s + lk][lr];
        if (s < 4) y0 = __builtin_amdgcn_mfma_f64_16x16x4f64(sT[lr][4 * s + lk], x, y0, 0, 0, 0);
        y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(sT[16 + lr][4 * s + lk], x, y1, 0, 0, 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + 4 * i + lk;
        if (r < D) L[(int64_t)r * D + n] = -y0[i];
        if (r + 16 < D) L[(int64_t)(r + 16) * D + n] = -y1[i];
      }
    }
    df_sync();
  }
}

void launch_dense_factor(const NutsBuffers& B, int* failed, hipStream_t st) {
  hipLaunchKernelGGL(dense_factor_kernel, dim3(B.C), dim3(64 * DF_W), 0, st, B, failed);
}

}  // namespace nutsgpu
