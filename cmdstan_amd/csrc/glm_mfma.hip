// Batched logistic-regression gradient on FP64 matrix cores (gfx950), D <= 128.
//
// For a tile of rows and 16 points per wave (v_mfma_f64_16x16x4):
//   phase 1  Eta = X_tile . Q^T           M = rows, N = points, K = D
//   pointwise R = sigmoid(Eta) - y, lp += y.Eta - log1p(e^Eta)   (in registers)
//   phase 2  G^T += R^T . X_tile           M = points, N = D, K = rows
// The 16x16x4 f64 result layout puts element (4i + l/16, l%16) in register i of
// lane l.  Phase 2 walks the rows of the tile in the order (block rb, register
// i, lane group l/16), so the A operand of each phase-2 step is exactly register
// i of the phase-1 accumulator of block rb: R never leaves the registers.  The
// B operand of phase 2 reads X in that same row order from the LDS tile that
// phase 1 used.
//
// Two ways to share a block's four waves:
//   SPLIT = 1  64 points, 16 per wave, on a common 32-row tile, double-buffered
//              in LDS (more than 16 points)
//   SPLIT = 4  16 points, the waves on row tiles of their own (16 rows each, in
//              wave-private LDS: no barriers), summed at the end (at most 16
//              points: three of four waves would multiply padding)
// The next tile's loads are issued before the current tile's products and wait
// in registers (2 D / 16 doubles per thread) until they are done.
//
// The step counts are template parameters (DT 16-column tiles, KS = 4 DT - R
// four-column steps), so the products are straight-line code whose operand
// reads run ahead of them.  With runtime counts every step was a branch, an LDS
// read waited for at once, and -- the tile being copied straight to LDS -- a
// wait for the whole copy of the next tile: 45-50% of the FP64 matrix peak at
// N = 100000, D = 100, 1024 points.
//
// Work split: blocks own (row chunk, 64-point group); the linear block id is
// remapped so that the groups sharing one row chunk run on the same XCD and
// share its L2.  Chunk partials go to a workspace reduced in fixed order
// (deterministic, no atomics).
#include "device_common.h"
#include "glm_split.h"
#include "launch.h"

namespace nutsgpu {

typedef double d4 __attribute__((ext_vector_type(4)));


#define GM_TC 64    // points per group of the work split
#define GM_KMAX 128 // D capacity

// The residual and the log-likelihood of one observation; a row past the chunk
// (live false) counts as zero.  lp takes y e - max(e, 0), lg the log1p term (as
// a factor): the vector unit's FP64 work shares its pipes with the FP64 matrix
// products, so these operations add to the products' time instead of hiding
// behind it -- a series of log1p per observation was a third of them.
__device__ __forceinline__ double gm_residual(double e, double yy, bool live, double& lp, LogProduct& lg) {
  const double t = exp(-fabs(e));
  const double d = 1.0 + t;
  const double r = (e >= 0.0 ? 1.0 : t) * recip_small(d) - yy;
  lp += live ? yy * e - (e > 0.0 ? e : 0.0) : 0.0;
  if (live) lg.times(t, d);
  return live ? r : 0.0;
}

template <int DT, int R, int SPLIT>
__global__ void __launch_bounds__(256, 2)
glm_mfma_f64(const double* __restrict__ X, const double* __restrict__ y, int N, int D, int total_blocks,
             const double* __restrict__ Q, int64_t ldq, int C, const int* __restrict__ need,
             const int* __restrict__ idx, const int* __restrict__ n_active, double* __restrict__ Wg,
             double* __restrict__ Wlp) {
  constexpr int KS = 4 * DT - R;              // phase-1 steps
  constexpr int XS = 16 * DT + 2;             // LDS row stride
  constexpr int TR = SPLIT == 1 ? 32 : 16;    // rows per tile
  constexpr int RB = TR / 16;
  constexpr int STEP = SPLIT == 1 ? 32 : 64;  // rows per iteration of the block
  constexpr int FR = SPLIT == 1 ? 2 : 4;      // prefetched rows per thread
  __shared__ double sX[SPLIT == 1 ? 2 : 4][TR * XS];
  __shared__ double sY[SPLIT == 1 ? 2 : 4][TR];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int lr = l & 15;   // m/n index inside a 16-wide tile
  const int lk = l >> 4;   // k index inside a 4-deep step

  // XCD-aware mapping: consecutive linear ids go to consecutive XCDs.
  const ActiveChains act(need, idx, n_active, C);
  const int n_act = act.n;
  const GlmSplit sp = glm_split(n_act, N, total_blocks);
  const int lin = blockIdx.x;
  const int xcd = lin & 7;
  const int j = lin >> 3;
  const int chunk = xcd + 8 * (j / sp.groups);
  const int group = j % sp.groups;
  if (chunk >= sp.chunks || group * GM_TC >= n_act) return;

  const int c0 = group * GM_TC + (SPLIT == 1 ? 16 * w : 0);  // this wave's 16 positions
  // phase-1 B operand for all k-steps: Q[c0 + lr][4 ks + lk]
  double qreg[KS];
  {
    const int pos = c0 + lr;
    const bool live = pos < n_act;
    const double* qr = Q + (int64_t)act.at(pos) * ldq;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int k = 4 * ks + lk;
      const double v = qr[k < D ? k : 0];
      qreg[ks] = live && k < D ? v : 0.0;
    }
  }
  d4 gacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) gacc[t] = d4{0, 0, 0, 0};
  double lp = 0.0;
  LogProduct lg;
  int tile = 0;
  const int n_begin = chunk * sp.rows;
  const int n_end = min(N, n_begin + sp.rows);

  // prefetch: 16 lanes cover 16 consecutive columns of a row (128-byte
  // segments); rows and columns outside read a clamped address and count as zero
  const int pr = SPLIT == 1 ? tid >> 4 : lk;      // first row of this thread in the tile
  constexpr int PS = SPLIT == 1 ? 16 : 4;         // its row step
  const int roff = SPLIT == 1 ? 0 : 16 * w;       // the wave's rows inside an iteration
  double xr[FR][DT], yr = 0.0;
  auto fetch = [&](int nb) {
#pragma unroll
    for (int m = 0; m < FR; ++m) {
      const int n = nb + roff + pr + PS * m;
      const double* row = X + (int64_t)(n < n_end ? n : n_end - 1) * D;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const int k = 16 * t + lr;
        const double v = row[t < DT - 1 || k < D ? k : 0];
        xr[m][t] = n < n_end && (t < DT - 1 || k < D) ? v : 0.0;
      }
    }
    const int ny = nb + roff + (SPLIT == 1 ? (tid & 31) : lr);
    yr = ny < n_end ? y[ny] : 0.0;
  };
  auto stash = [&](int b) {
    double* sx = sX[b];
#pragma unroll
    for (int m = 0; m < FR; ++m)
#pragma unroll
      for (int t = 0; t < DT; ++t) sx[(pr + PS * m) * XS + 16 * t + lr] = xr[m][t];
    if (SPLIT == 1 ? tid < TR : l < TR) sY[b][SPLIT == 1 ? tid : l] = yr;
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
    const double* sx = sX[b];
    const double* sy = sY[b];
    d4 eta[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) eta[rb] = d4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        eta[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(sx[(16 * rb + lr) * XS + 4 * ks + lk], qreg[ks], eta[rb], 0, 0, 0);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rr = 16 * rb + 4 * i + lk;
        eta[rb][i] = gm_residual(eta[rb][i], sy[rr], nb + roff + rr < n_end, lp, lg);
      }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double* xrow = sx + (16 * rb + 4 * i + lk) * XS + lr;
#pragma unroll
        for (int t = 0; t < DT; ++t)
          gacc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(eta[rb][i], xrow[16 * t], gacc[t], 0, 0, 0);
      }
    if (more) {
      if (++tile % 64 == 0) lg.fold();   // at most 512 factors since the last
      if constexpr (SPLIT == 1) b ^= 1;  // the other buffer: its readers passed this iteration's barrier
      else {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      stash(b);
    }
  }

  lp -= lg.log_value();
  lp += __shfl_xor(lp, 16, 64);
  lp += __shfl_xor(lp, 32, 64);
  if constexpr (SPLIT == 4) {
    // the four waves' sums: tile by tile through LDS, wave 0 + 1 + 2 + 3
    __shared__ double red[4][256];
    __shared__ double redlp[4][16];
    if (lk == 0) redlp[w][lr] = lp;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) red[w][64 * i + l] = gacc[t][i];
      __syncthreads();
      const int pos = c0 + (tid >> 4), d = 16 * t + (tid & 15);  // element tid: point tid / 16, column tid % 16
      if (pos < n_act && d < D)
        Wg[((int64_t)chunk * sp.stride + pos) * D + d] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
    }
    if (tid < 16 && c0 + tid < n_act)
      Wlp[(int64_t)chunk * sp.stride + c0 + tid] =
          ((redlp[0][tid] + redlp[1][tid]) + redlp[2][tid]) + redlp[3][tid];
  } else {
    // gacc[t] register i of lane l = G[chain c0 + 4i + lk][d 16t + lr]; lanes l,
    // l + 16, l + 32, l + 48 hold the same chain's lp
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int d = 16 * t + lr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pos = c0 + 4 * i + lk;
        if (pos < n_act && d < D) Wg[((int64_t)chunk * sp.stride + pos) * D + d] = gacc[t][i];
      }
    }
    if (lk == 0 && c0 + lr < n_act) Wlp[(int64_t)chunk * sp.stride + c0 + lr] = lp;
  }
}

// G and V of every point from the chunk partials: 64 columns x 8 chunk slices
// per block, a fixed order (slice z takes chunks z, z + 8, ...), eight loads in
// flight per thread.  A few points have few blocks and many chunks: one thread
// per column walking all chunks took 8.0 us at 160 chunks.
__global__ void __launch_bounds__(512)
glm_mfma_reduce(const double* __restrict__ Wg, const double* __restrict__ Wlp, int N, int total_blocks, int C, int D,
                double s2inv, const double* __restrict__ Q, int64_t ldq, const int* __restrict__ need,
                const int* __restrict__ idx, const int* __restrict__ n_active, long long* __restrict__ tally,
                double sign, double* __restrict__ G, double* __restrict__ V) {
  __shared__ double red[8][64];
  const int pos = blockIdx.x;
  const ActiveChains act(need, idx, n_active, C);
  const int n_act = act.n;
  if (pos >= n_act) return;
  const GlmSplit sp = glm_split(n_act, N, total_blocks);
  const int c = __builtin_amdgcn_readfirstlane(act.at(pos));
  if (tally && pos == 0 && blockIdx.y == 0 && threadIdx.x == 0) *tally += n_act;
  const double* q = Q + (int64_t)c * ldq;
  double* g = G + (int64_t)c * ldq;
  const int lane = threadIdx.x & 63, z = threadIdx.x >> 6;
  const int k = blockIdx.y * 64 + lane;
  double s = 0.0;
  if (k < D) {
#pragma unroll 8
    for (int ch = z; ch < sp.chunks; ch += 8) s += Wg[((int64_t)ch * sp.stride + pos) * D + k];
  }
  red[z][lane] = s;
  __syncthreads();
  if (z == 0 && k < D) {
    double t = 0.0;
#pragma unroll
    for (int v = 0; v < 8; v += 2) t += red[v][lane] + red[v + 1][lane];
    g[k] = sign * (t + s2inv * q[k]);
  }
  if (blockIdx.y == 0 && z == 1) {
    double lpv = 0.0, pr = 0.0;
    for (int ch = lane; ch < sp.chunks; ch += 64) lpv += Wlp[(int64_t)ch * sp.stride + pos];
    for (int i = lane; i < D; i += 64) pr += q[i] * q[i];
    lpv = wave_sum(lpv);
    pr = wave_sum(pr);
    if (lane == 0) V[c] = -sign * (lpv - 0.5 * s2inv * pr);
  }
}

// Active-chain list for the lockstep gradient: idx[0..n) = chains with need[c]
// set, in chain order (single-block scan, deterministic); clears need[].
__global__ void __launch_bounds__(1024) compact_active(int* __restrict__ need, int C, int* __restrict__ idx,
                                                       int* __restrict__ n_active, long long* __restrict__ tally) {
  __shared__ int wsum[16];
  __shared__ int base;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  if (t == 0) base = 0;
  __syncthreads();
  for (int c0 = 0; c0 < C; c0 += 1024) {
    const int c = c0 + t;
    const int f = (c < C && need[c]) ? 1 : 0;
    if (c < C) need[c] = 0;
    int x = f;  // inclusive wave scan
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    int off = base;
    for (int k = 0; k < wv; ++k) off += wsum[k];
    if (f) idx[off + x - 1] = c;
    __syncthreads();
    if (t == 1023) {
      int tot = 0;
      for (int k = 0; k < 16; ++k) tot += wsum[k];
      base += tot;
    }
    __syncthreads();
  }
  if (t == 0) {
    *n_active = base;
    if (tally) *tally += base;
  }
}

void launch_compact_active(int* need, int C, int* idx, int* n_active, long long* tally, hipStream_t st) {
  hipLaunchKernelGGL(compact_active, dim3(1), dim3(1024), 0, st, need, C, idx, n_active, tally);
}

GlmPlan glm_mfma_plan(int N, int C, int D, int num_cus, int blocks_per_cu) {
  GlmPlan p;
  // blocks_per_cu resident blocks per CU (2 unless tuned), and at least 8 row
  // chunks per chain group
  const int groups = (C + GM_TC - 1) / GM_TC;
  int tb = (blocks_per_cu > 0 ? blocks_per_cu : 2) * (num_cus > 0 ? num_cus : 256);
  if (tb < 8 * groups) tb = 8 * groups;
  p.total_blocks = (tb + 7) & ~7;
  const GlmSplit full = glm_split(C, N, p.total_blocks);
  p.ngroups = full.groups;
  p.nchunks = full.chunks;
  p.rows_per_chunk = full.rows;
  // partials of any launch: chunks * stride <= total_blocks * 64 positions
  p.work_doubles = (size_t)p.total_blocks * GM_TC * D + (size_t)p.total_blocks * GM_TC;
  return p;
}

template <int DT, int R>
static void gm_launch(const GlmArgs& a, const GlmPlan& p, double* Wg, double* Wlp, hipStream_t st) {
  // at most 16 points: the waves split the rows (see the top of the file)
  if (a.C <= 16)
    hipLaunchKernelGGL((glm_mfma_f64<DT, R, 4>), dim3(p.total_blocks), dim3(256), 0, st, a.X, a.y, a.N, a.D,
                       p.total_blocks, a.Q, a.ldq, a.C, a.need, a.idx, a.n_active, Wg, Wlp);
  else
    hipLaunchKernelGGL((glm_mfma_f64<DT, R, 1>), dim3(p.total_blocks), dim3(256), 0, st, a.X, a.y, a.N, a.D,
                       p.total_blocks, a.Q, a.ldq, a.C, a.need, a.idx, a.n_active, Wg, Wlp);
}

template <int DT>
static void gm_launch_tiles(const GlmArgs& a, const GlmPlan& p, double* Wg, double* Wlp, hipStream_t st) {
  switch (4 * DT - (a.D + 3) / 4) {  // four-column steps the last tile leaves out
    case 0: gm_launch<DT, 0>(a, p, Wg, Wlp, st); break;
    case 1: gm_launch<DT, 1>(a, p, Wg, Wlp, st); break;
    case 2: gm_launch<DT, 2>(a, p, Wg, Wlp, st); break;
    default: gm_launch<DT, 3>(a, p, Wg, Wlp, st); break;
  }
}

int glm_grad_mfma_f64(const GlmArgs& a, const GlmPlan& p, hipStream_t st) {
  if (a.D > GM_KMAX || a.D < 1) return 1;
  double* Wg = a.work;
  double* Wlp = a.work + (size_t)p.total_blocks * GM_TC * a.D;
  if (a.ev_begin) (void)hipEventRecord(a.ev_begin, st);
  switch ((a.D + 15) / 16) {
    case 1: gm_launch_tiles<1>(a, p, Wg, Wlp, st); break;
    case 2: gm_launch_tiles<2>(a, p, Wg, Wlp, st); break;
    case 3: gm_launch_tiles<3>(a, p, Wg, Wlp, st); break;
    case 4: gm_launch_tiles<4>(a, p, Wg, Wlp, st); break;
    case 5: gm_launch_tiles<5>(a, p, Wg, Wlp, st); break;
    case 6: gm_launch_tiles<6>(a, p, Wg, Wlp, st); break;
    case 7: gm_launch_tiles<7>(a, p, Wg, Wlp, st); break;
    default: gm_launch_tiles<8>(a, p, Wg, Wlp, st); break;
  }
  if (a.ev_end) (void)hipEventRecord(a.ev_end, st);
  glm_reduce_launch(a, p, st);
  return 0;
}

void glm_reduce_launch(const GlmArgs& a, const GlmPlan& p, hipStream_t st) {
  double* Wg = a.work;
  double* Wlp = a.work + (size_t)p.total_blocks * GM_TC * a.D;
  hipLaunchKernelGGL(glm_mfma_reduce, dim3(a.C, (a.D + 63) / 64), dim3(512), 0, st, Wg, Wlp, a.N, p.total_blocks, a.C,
                     a.D, a.s2inv, a.Q, a.ldq, a.need, a.idx, a.n_active, a.tally, a.sign, a.G,
                     a.V);
}

}  // namespace nutsgpu
