// Batched logistic-regression gradient with the contraction on FP32 matrix
// cores (v_mfma_f32_16x16x4f32, FP32 accumulation) and X stored in FP32 or
// BF16 (converted to FP32 on its way into LDS).  The per-observation terms are
// formed in FP32 from the FP32 linear predictor and the per-chain log density
// is summed in FP64; chunk partials of the gradient are reduced in FP64, so V
// and ∇V reach the FP64 sampler with an error set by FP32 rounding of the
// products and terms (stated against FP64 in the tests).
//
// Same structure as the FP64 kernel: phase 1 Eta = X·Qᵀ, pointwise R, phase 2
// Gᵀ += Rᵀ·X with the K order of phase 2 permuted so its A operand is the
// phase-1 accumulator; a block owns (row chunk, 64 points), four waves of 16
// points on common 32-row tiles, or for at most 16 points four waves on row
// tiles of their own; the next tile's loads are in flight during the products,
// and the tile count is a template parameter, so the products are straight-line
// code (with runtime counts each step was a branch and a waited-for LDS read).
// Phase 1 takes its columns in the order 16 q + 4 (l / 16) + i: a lane's four
// A operands of a 16-column tile are one 16-byte LDS read (row stride 16 DT + 4
// floats, an odd number of 16-byte slots: no bank conflicts).
// Bound: the FP32 matrix rate and, beside it, the terms' vector work: at N =
// 100000, D = 100, 1024 points 494 us of 275 at the rate a large product reaches
// (2.86 ms before, with scalar LDS reads behind a branch per step and tiles loaded
// between two barriers); 50000 x 128 at 16 points 224 -> 19 us.
#include <hip/hip_bf16.h>

#include "device_common.h"
#include "glm_split.h"
#include "launch.h"

namespace nutsgpu {

typedef float f4 __attribute__((ext_vector_type(4)));

#define GF_TC 64
#define GF_KMAX 128
#define GF_FOLD 8

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(unsigned short b) { return __uint_as_float(((unsigned)b) << 16); }

// Register i of lane l in a 16x16 f32 result is row 4 (l / 16) + i, column l % 16.
template <typename XT, int DT, int SPLIT>
__global__ void __launch_bounds__(256, 2)
glm_mfma_f32(const XT* __restrict__ X, const double* __restrict__ y, int N, int D, int total_blocks,
             const double* __restrict__ Q, int64_t ldq, int C, const int* __restrict__ idx,
             const int* __restrict__ n_active, double* __restrict__ Wg, double* __restrict__ Wlp) {
  constexpr int XS = 16 * DT + 4;             // LDS row stride in floats
  constexpr int TR = SPLIT == 1 ? 32 : 16;    // rows per tile
  constexpr int RB = TR / 16;
  constexpr int STEP = SPLIT == 1 ? 32 : 64;  // rows per iteration of the block
  constexpr int FR = SPLIT == 1 ? 2 : 4;      // prefetched rows per thread
  constexpr int NB = SPLIT == 1 ? 2 : 4;
  __shared__ __attribute__((aligned(16))) float sX[NB][TR * XS];
  __shared__ float sY[NB][TR];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int lr = l & 15;
  const int lk = l >> 4;

  const int n_act = idx ? *n_active : C;
  const GlmSplit sp = glm_split(n_act, N, total_blocks);
  const int lin = blockIdx.x;
  const int xcd = lin & 7;
  const int j = lin >> 3;
  const int chunk = xcd + 8 * (j / sp.groups);
  const int group = j % sp.groups;
  if (chunk >= sp.chunks || group * GF_TC >= n_act) return;

  const int c0 = group * GF_TC + (SPLIT == 1 ? 16 * w : 0);
  float qreg[4 * DT];  // phase-1 B operand: Q[c0 + lr][16 t + 4 lk + i]
  {
    const int pos = c0 + lr;
    const int c = pos < n_act ? (idx ? idx[pos] : pos) : -1;
    const double* qr = Q + (int64_t)(c < 0 ? 0 : c) * ldq;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 16 * t + 4 * lk + i;
        const double v = qr[k < D ? k : 0];
        qreg[4 * t + i] = c >= 0 && k < D ? (float)v : 0.0f;
      }
  }
  // gacc sums GF_FOLD tiles and is then added to gsum: a chunk of thousands of
  // rows in one FP32 chain rounds noticeably more
  f4 gacc[DT], gsum[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) gacc[t] = gsum[t] = f4{0, 0, 0, 0};
  double lp = 0.0;
  int tile = 0;
  const int n_begin = chunk * sp.rows;
  const int n_end = min(N, n_begin + sp.rows);

  // prefetch: 16 lanes cover 16 consecutive columns of a row; rows and columns
  // outside read a clamped address and count as zero
  const int pr = SPLIT == 1 ? tid >> 4 : lk;
  constexpr int PS = SPLIT == 1 ? 16 : 4;
  const int roff = SPLIT == 1 ? 0 : 16 * w;
  XT xr[FR][DT];
  double yr = 0.0;
  auto fetch = [&](int nb) {
#pragma unroll
    for (int m = 0; m < FR; ++m) {
      const int n = nb + roff + pr + PS * m;
      const XT* row = X + (int64_t)(n < n_end ? n : n_end - 1) * D;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const int k = 16 * t + lr;
        const XT v = row[t < DT - 1 || k < D ? k : 0];
        xr[m][t] = n < n_end && (t < DT - 1 || k < D) ? v : XT(0);
      }
    }
    const int ny = nb + roff + (SPLIT == 1 ? (tid & 31) : lr);
    yr = ny < n_end ? y[ny] : 0.0;
  };
  auto stash = [&](int b) {
    float* sx = sX[b];
#pragma unroll
    for (int m = 0; m < FR; ++m)
#pragma unroll
      for (int t = 0; t < DT; ++t) sx[(pr + PS * m) * XS + 16 * t + lr] = to_f32(xr[m][t]);
    if (SPLIT == 1 ? tid < TR : l < TR) sY[b][SPLIT == 1 ? tid : l] = (float)yr;
  };
  int b = SPLIT == 1 ? 0 : w;
  if (n_begin < n_end) {
    fetch(n_begin);
    stash(b);
  }
  for (int nb = n_begin; nb < n_end; nb += STEP) {
    if constexpr (SPLIT == 1) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    const bool more = nb + STEP < n_end;
    if (more) fetch(nb + STEP);
    const float* sx = sX[b];
    const float* sy = sY[b];
    f4 eta[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) eta[rb] = f4{0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      f4 xa[RB];
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) xa[rb] = *reinterpret_cast<const f4*>(sx + (16 * rb + lr) * XS + 16 * t + 4 * lk);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          eta[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[rb][i], qreg[4 * t + i], eta[rb], 0, 0, 0);
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // terms in FP32 from the FP32 linear predictor, summed in FP64
        const int rr = 16 * rb + 4 * lk + i;
        const bool live = nb + roff + rr < n_end;
        const float e = eta[rb][i], yy = sy[rr];
        const float t = __expf(-fabsf(e));
        const float l1p = t < 1e-4f ? t * (1.0f - 0.5f * t) : __logf(1.0f + t);
        lp += live ? (double)(yy * e - ((e > 0.0f ? e : 0.0f) + l1p)) : 0.0;
        eta[rb][i] = live ? (e >= 0.0f ? 1.0f : t) / (1.0f + t) - yy : 0.0f;
      }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* xrow = sx + (16 * rb + 4 * lk + i) * XS + lr;
#pragma unroll
        for (int t = 0; t < DT; ++t)
          gacc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(eta[rb][i], xrow[16 * t], gacc[t], 0, 0, 0);
      }
    if (++tile % GF_FOLD == 0 || !more) {
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        gsum[t] += gacc[t];
        gacc[t] = f4{0, 0, 0, 0};
      }
    }
    if (more) {
      if constexpr (SPLIT == 1) b ^= 1;  // the other buffer: its readers passed this iteration's barrier
      else {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      stash(b);
    }
  }

  lp += __shfl_xor(lp, 16, 64);
  lp += __shfl_xor(lp, 32, 64);
  if constexpr (SPLIT == 4) {
    // the four waves' sums in FP64: tile by tile through LDS, wave 0 + 1 + 2 + 3
    __shared__ double red[4][256];
    __shared__ double redlp[4][16];
    if (lk == 0) redlp[w][lr] = lp;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) red[w][16 * (4 * lk + i) + lr] = (double)gsum[t][i];
      __syncthreads();
      const int pos = c0 + (tid >> 4), d = 16 * t + (tid & 15);  // element tid: point tid / 16, column tid % 16
      if (pos < n_act && d < D)
        Wg[((int64_t)chunk * sp.stride + pos) * D + d] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
    }
    if (tid < 16 && c0 + tid < n_act)
      Wlp[(int64_t)chunk * sp.stride + c0 + tid] =
          ((redlp[0][tid] + redlp[1][tid]) + redlp[2][tid]) + redlp[3][tid];
  } else {
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int d = 16 * t + lr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pos = c0 + 4 * lk + i;
        if (pos < n_act && d < D) Wg[((int64_t)chunk * sp.stride + pos) * D + d] = (double)gsum[t][i];
      }
    }
    if (lk == 0 && c0 + lr < n_act) Wlp[(int64_t)chunk * sp.stride + c0 + lr] = lp;
  }
}

__global__ void glm_to_f32(const double* __restrict__ X, float* __restrict__ Y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) Y[i] = (float)X[i];
}
// round to nearest even bf16
__global__ void glm_to_bf16(const double* __restrict__ X, unsigned short* __restrict__ Y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const unsigned u = __float_as_uint((float)X[i]);
    const unsigned r = u + 0x7FFFu + ((u >> 16) & 1u);
    Y[i] = (unsigned short)(r >> 16);
  }
}

void glm_convert_x(const double* X, void* out, int64_t n, int precision, hipStream_t st) {
  const dim3 grid((unsigned)((n + 255) / 256)), blk(256);
  if (precision == 1) hipLaunchKernelGGL(glm_to_f32, grid, blk, 0, st, X, (float*)out, n);
  else hipLaunchKernelGGL(glm_to_bf16, grid, blk, 0, st, X, (unsigned short*)out, n);
}

template <typename XT, int DT>
static void gf_launch(const GlmArgs& a, const GlmPlan& p, const XT* X, double* Wg, double* Wlp, hipStream_t st) {
  // at most 16 points: the waves split the rows (three of four would multiply padding)
  if (a.C <= 16)
    hipLaunchKernelGGL((glm_mfma_f32<XT, DT, 4>), dim3(p.total_blocks), dim3(256), 0, st, X, a.y, a.N, a.D,
                       p.total_blocks, a.Q, a.ldq, a.C, a.idx, a.n_active, Wg, Wlp);
  else
    hipLaunchKernelGGL((glm_mfma_f32<XT, DT, 1>), dim3(p.total_blocks), dim3(256), 0, st, X, a.y, a.N, a.D,
                       p.total_blocks, a.Q, a.ldq, a.C, a.idx, a.n_active, Wg, Wlp);
}

template <typename XT>
static void gf_launch_tiles(const GlmArgs& a, const GlmPlan& p, const void* Xlow, double* Wg, double* Wlp,
                            hipStream_t st) {
  const XT* X = (const XT*)Xlow;
  switch ((a.D + 15) / 16) {
    case 1: gf_launch<XT, 1>(a, p, X, Wg, Wlp, st); break;
    case 2: gf_launch<XT, 2>(a, p, X, Wg, Wlp, st); break;
    case 3: gf_launch<XT, 3>(a, p, X, Wg, Wlp, st); break;
    case 4: gf_launch<XT, 4>(a, p, X, Wg, Wlp, st); break;
    case 5: gf_launch<XT, 5>(a, p, X, Wg, Wlp, st); break;
    case 6: gf_launch<XT, 6>(a, p, X, Wg, Wlp, st); break;
    case 7: gf_launch<XT, 7>(a, p, X, Wg, Wlp, st); break;
    default: gf_launch<XT, 8>(a, p, X, Wg, Wlp, st); break;
  }
}

// The reduce kernel of the FP64 path sums the chunk partials in FP64.
int glm_grad_mfma_f32(const GlmArgs& a, const GlmPlan& p, const void* Xlow, int precision, hipStream_t st) {
  if (a.D > GF_KMAX || a.D < 1) return 1;
  double* Wg = a.work;
  double* Wlp = a.work + (size_t)p.total_blocks * GF_TC * a.D;
  if (a.ev_begin) (void)hipEventRecord(a.ev_begin, st);
  if (precision == 1) gf_launch_tiles<float>(a, p, Xlow, Wg, Wlp, st);
  else gf_launch_tiles<unsigned short>(a, p, Xlow, Wg, Wlp, st);
  if (a.ev_end) (void)hipEventRecord(a.ev_end, st);
  glm_reduce_launch(a, p, st);
  return 0;
}

}  // namespace nutsgpu
