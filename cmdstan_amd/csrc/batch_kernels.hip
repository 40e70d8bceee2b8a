// Small kernels around a sampling run: its start metric, the layout of its
// results (what the host did element by element).
#include "device_common.h"
#include "launch.h"

namespace nutsgpu {

// M[c][j][i] = A[c][i][j] for C contiguous D x D blocks (32 x 32 tiles through
// LDS); *bad set when an element is not finite
__global__ void __launch_bounds__(256) metric_transpose_kernel(const double* __restrict__ A, double* __restrict__ M,
                                                               int D, int* __restrict__ bad) {
  __shared__ double t[32][33];
  const int64_t base = (int64_t)blockIdx.z * D * D;
  const int j0 = blockIdx.x * 32, i0 = blockIdx.y * 32;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  bool ok = true;
  for (int r = y; r < 32; r += 8) {
    const int i = i0 + r, j = j0 + x;
    if (i < D && j < D) {
      const double v = A[base + (int64_t)i * D + j];
      ok = ok && isfinite(v);
      t[r][x] = v;
    }
  }
  if (bad && !ok) *bad = 1;
  __syncthreads();
  for (int r = y; r < 32; r += 8) {
    const int j = j0 + r, i = i0 + x;
    if (i < D && j < D) M[base + (int64_t)j * D + i] = t[x][r];
  }
}

void launch_metric_transpose(const double* A, double* M, int C, int D, int* bad, hipStream_t st) {
  const int n = (D + 31) / 32;
  for (int c = 0; c < C; c += 32768) {
    const int64_t o = (int64_t)c * D * D;
    hipLaunchKernelGGL(metric_transpose_kernel, dim3(n, n, C - c < 32768 ? C - c : 32768), dim3(256), 0, st, A + o,
                       M + o, D, bad);
  }
}

// identity blocks of the chains' dimensions at moff
__global__ void __launch_bounds__(256) metric_identity_kernel(double* __restrict__ M, const int* __restrict__ D,
                                                              const int64_t* __restrict__ moff) {
  const int c = blockIdx.y, d = D[c];
  double* m = M + moff[c];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < (int64_t)d * d; i += (int64_t)gridDim.x * 256)
    m[i] = i % d == i / d ? 1.0 : 0.0;
}

void launch_metric_identity(double* M, const int* D, const int64_t* moff, int C, int maxD, hipStream_t st) {
  const int bx = (int)(((int64_t)maxD * maxD + 256 * 16 - 1) / (256 * 16));
  for (int c = 0; c < C; c += 32768)
    hipLaunchKernelGGL(metric_identity_kernel, dim3(bx, C - c < 32768 ? C - c : 32768), dim3(256), 0, st, M, D + c,
                       moff + c);
}

template <class T>
__global__ void fill_kernel(T* p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

void launch_fill(double* p, int64_t n, double v, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(fill_kernel<double>, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, st, p, n, v);
}
void launch_fill(float* p, int64_t n, float v, hipStream_t st) {
  if (n > 0) hipLaunchKernelGGL(fill_kernel<float>, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, st, p, n, v);
}

// rows of D[c] values at src + off[c], packed at out + to[c]
template <class T>
__global__ void __launch_bounds__(256) pack_rows_kernel(const T* __restrict__ src, const int64_t* __restrict__ off,
                                                        const int* __restrict__ D, const int64_t* __restrict__ to,
                                                        double* __restrict__ out) {
  const int c = blockIdx.x;
  for (int i = threadIdx.x; i < D[c]; i += 256) out[to[c] + i] = (double)src[off[c] + i];
}

void launch_pack_rows(const void* src, bool f32, const int64_t* off, const int* D, const int64_t* to, int C,
                      double* out, hipStream_t st) {
  if (f32)
    hipLaunchKernelGGL(pack_rows_kernel<float>, dim3(C), dim3(256), 0, st, (const float*)src, off, D, to, out);
  else hipLaunchKernelGGL(pack_rows_kernel<double>, dim3(C), dim3(256), 0, st, (const double*)src, off, D, to, out);
}

}  // namespace nutsgpu
