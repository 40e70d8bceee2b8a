// Batched logistic-regression gradient on FP64 matrix cores for 128 < D <= 1024
// (v_mfma_f64_16x16x4): one pass over X, no residual matrix in memory.
//
// A block takes 16 or 32 points and a chunk of rows; its W waves split the
// columns, tiles of 16 dealt round (up to TW a wave).  Per 16-row tile:
//   phase 1  every wave: its columns' share of Eta = X Q^T (M = rows, N = points)
//   sum      the W partial Etas through LDS, one result register per wave;
//            R = sigmoid(Eta) - y and the lp terms, R back through LDS
//   phase 2  every wave: G^T[:, its columns] += R^T X (M = points, K = rows)
// A wave's X tile is private (it reads the columns it owns in both phases), so
// it is staged in its own LDS strip without block barriers, and the next
// tile's loads are in flight (in registers) during the products.  Result
// register i of lane l is row 4i + l/16, column l%16, which is the A operand of
// phase-2 step i: R needs no shuffles.
//
// Bound: FP64 matrix cores (a 16x16x4 product occupies a SIMD for 64 cycles;
// its operands are one 8-byte LDS read per lane), then the two block barriers
// per tile.  Splitting the columns over the waves, not the points, keeps 16 or
// 32 points enough to fill a block, so a few points still spread over every CU
// by row chunks.  Measured, N = 10000, D = 500: 64 points 24.0 ms with a wave
// per point (LogisticFn) -> 57 us (51.6 us in this kernel, 24.8 TFLOP/s), 4
// points 36 us, 1024 points 601 us (34 TFLOP/s).  One block of eight waves per
// CU: two blocks of four waves (8 tiles each) spilled and took 98 us, and
// skipping the tiles past D by branches cost 90 us (the operand reads no
// longer overlap the products), so the tile count is a template parameter and
// at most one tile per wave is padding.
#include "device_common.h"
#include "glm_wide.h"

namespace nutsgpu {

typedef double d4 __attribute__((ext_vector_type(4)));

namespace {

struct GwSplit {
  int groups, chunks, rows;  // groups of gp points, row chunks, rows per chunk (multiple of 16)
};

__host__ __device__ inline GwSplit gw_split(int n_act, int N, int total_blocks, int max_chunks, int gp) {
  GwSplit s;
  s.groups = n_act > 0 ? (n_act + gp - 1) / gp : 1;
  int ch = total_blocks / s.groups;
  if (ch > max_chunks) ch = max_chunks;
  // whole chunks per XCD when there is more than one chunk for each
  if (ch > 8) ch &= ~7;
  const int tiles = (N + 15) / 16;
  if (ch > tiles) ch = tiles;
  if (ch < 1) ch = 1;
  s.rows = (tiles + ch - 1) / ch * 16;
  s.chunks = tiles > 0 ? (tiles * 16 + s.rows - 1) / s.rows : 1;
  if (s.rows < 16) s.rows = 16;
  return s;
}

}  // namespace

template <int W, int TW, int NG>
__global__ void __launch_bounds__(64 * W, 2)
glm_wide_f64(GlmArgs a, int total_blocks, int max_chunks, double* __restrict__ Wg, double* __restrict__ Wlp) {
  constexpr int COLS = 16 * TW;
  constexpr int XS = COLS + 2;
  constexpr int GP = 16 * NG;  // points per block
  __shared__ double sX[W][16 * XS];
  __shared__ double sE[W][NG * 256];
  __shared__ double sR[NG * 256];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, lr = l & 15, lk = l >> 4;
  const ActiveChains act(a.need, a.idx, a.n_active, a.C);
  const int n_act = act.n;
  const GwSplit sp = gw_split(n_act, a.N, total_blocks, max_chunks, GP);
  // blocks of one row chunk (all groups) on one XCD, so X is fetched once per L2
  const int lin = blockIdx.x;
  int chunk, group;
  if ((sp.chunks & 7) == 0) {
    const int j = lin >> 3;
    chunk = (lin & 7) + 8 * (j / sp.groups);
    group = j % sp.groups;
  } else {
    chunk = lin / sp.groups;
    group = lin % sp.groups;
  }
  if (chunk >= sp.chunks || group * GP >= n_act) return;

  const int N = a.N, D = a.D;
  const int p0 = group * GP;
  // this wave's columns: 16-column tiles w, w + W, ... (the last may lie past D)
  auto col0 = [&](int t) { return 16 * (w + W * t); };
  double qreg[NG][4 * TW];  // phase-1 B operand: Q[point 16 g + lr][col0(ks / 4) + 4 (ks % 4) + lk]
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int pos = p0 + 16 * g + lr;
    const bool live = pos < n_act;
    const double* q = a.Q + (int64_t)act.at(pos) * a.ldq;
#pragma unroll
    for (int ks = 0; ks < 4 * TW; ++ks) {
      const int k = col0(ks >> 2) + 4 * (ks & 3) + lk;
      qreg[g][ks] = (live && k < D) ? q[k] : 0.0;
    }
  }
  d4 gacc[NG][TW];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int t = 0; t < TW; ++t) gacc[g][t] = d4{0, 0, 0, 0};
  const int n_begin = chunk * sp.rows, n_end = min(N, n_begin + sp.rows);
  double* sx = sX[w];
  // prefetch register [s][t]: row 4 s + lk, column col0(t) + lr; rows and
  // columns outside read a clamped address and count as zero (no branches)
  double xr[4][TW];
  auto fetch = [&](int nb) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int n = nb + 4 * s + lk;
      const double* row = a.X + (int64_t)(n < n_end ? n : n_end - 1) * D;
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const int k = col0(t) + lr;
        const double v = row[k < D ? k : D - 1];
        xr[s][t] = (n < n_end && k < D) ? v : 0.0;
      }
    }
  };
  // the 4 NG result registers (register i of group g is item 4 g + i) go
  // round the waves: wave w finishes items w, w + W, ...
  constexpr int IT = (4 * NG + W - 1) / W;
  double lp[IT];
  LogProduct lg[IT];
#pragma unroll
  for (int m = 0; m < IT; ++m) lp[m] = 0.0;
  if (n_begin < n_end) fetch(n_begin);
  for (int nb = n_begin; nb < n_end; nb += 16) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < TW; ++t) sx[(4 * s + lk) * XS + 16 * t + lr] = xr[s][t];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (nb + 16 < n_end) fetch(nb + 16);
    // two accumulators in turn: consecutive products are independent
    d4 e0[2], e1[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) e0[g] = e1[g] = d4{0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < 4 * TW; ks += 2) {
      const double x0 = sx[lr * XS + 4 * ks + lk], x1 = sx[lr * XS + 4 * ks + 4 + lk];
#pragma unroll
      for (int g = 0; g < NG; ++g) e0[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(x0, qreg[g][ks], e0[g], 0, 0, 0);
#pragma unroll
      for (int g = 0; g < NG; ++g) e1[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1, qreg[g][ks + 1], e1[g], 0, 0, 0);
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) sE[w][256 * g + 64 * i + l] = e0[g][i] + e1[g][i];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < IT; ++m) {
      const int item = w + W * m;
      if (item < 4 * NG) {
        double e = 0.0;
#pragma unroll
        for (int v = 0; v < W; ++v) e += sE[v][64 * item + l];
        const int n = nb + 4 * (item & 3) + lk;
        double r = 0.0;
        if (n < n_end) {
          const double yy = a.y[n];
          const double t = exp(-fabs(e));
          const double d = 1.0 + t;
          lp[m] += yy * e - (e > 0.0 ? e : 0.0);
          lg[m].times(t, d);
          lg[m].fold();
          r = (e >= 0.0 ? 1.0 : t) * recip_small(d) - yy;
        }
        sR[64 * item + l] = r;
      }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      double r[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) r[g] = sR[256 * g + 64 * s + l];
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const double x = sx[(4 * s + lk) * XS + 16 * t + lr];
#pragma unroll
        for (int g = 0; g < NG; ++g)
          gacc[g][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[g], x, gacc[g][t], 0, 0, 0);
      }
    }
  }
  // gacc[g][t] register i = G[point 16 g + 4i + lk][col0(t) + lr]; a single chunk is the whole sum
  const bool whole = sp.chunks == 1;
  const int64_t base = (int64_t)chunk * (GP * sp.groups);
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = p0 + 16 * g + 4 * i + lk;
      const int64_t row = whole ? (int64_t)act.at(p) * a.ldq : 0;
      if (p >= n_act) continue;
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const int d = col0(t) + lr;
        if (d >= D) continue;
        if (whole) a.G[row + d] = a.sign * (gacc[g][t][i] + a.s2inv * a.Q[row + d]);
        else Wg[(base + p) * D + d] = gacc[g][t][i];
      }
    }
  // lanes l, l + 16, l + 32, l + 48 and the four items of a group hold the same points
  __syncthreads();
#pragma unroll
  for (int m = 0; m < IT; ++m) {
    const int item = w + W * m;
    double v = lp[m] - lg[m].log_value();
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (item < 4 * NG && lk == 0) sR[16 * item + lr] = v;
  }
  __syncthreads();
  if (tid < GP && p0 + tid < n_act) {
    const double* s = sR + 64 * (tid >> 4) + (tid & 15);
    Wlp[base + p0 + tid] = (s[0] + s[16]) + (s[32] + s[48]);
  }
}

// G and V of every point from the chunk partials: 64 columns x 8 chunk slices
// per block, a fixed order (slice z takes chunks z, z + 8, ...), sixteen loads
// in flight per thread
__global__ void __launch_bounds__(512)
glm_wide_reduce(GlmArgs a, int total_blocks, int max_chunks, int gp, const double* __restrict__ Wg, const double* __restrict__ Wlp) {
  __shared__ double red[8][64];
  const int pos = blockIdx.x;
  const ActiveChains act(a.need, a.idx, a.n_active, a.C);
  const int n_act = act.n;
  if (pos >= n_act) return;
  const GwSplit sp = gw_split(n_act, a.N, total_blocks, max_chunks, gp);
  const int64_t stride = gp * sp.groups;
  const int c = __builtin_amdgcn_readfirstlane(act.at(pos));
  if (a.tally && pos == 0 && blockIdx.y == 0 && threadIdx.x == 0) *a.tally += n_act;
  const double* q = a.Q + (int64_t)c * a.ldq;
  const int lane = threadIdx.x & 63, z = threadIdx.x >> 6;
  if (sp.chunks > 1) {
    const int k = blockIdx.y * 64 + lane;
    double s = 0.0;
    if (k < a.D) {
#pragma unroll 16
      for (int ch = z; ch < sp.chunks; ch += 8) s += Wg[(ch * stride + pos) * a.D + k];
    }
    red[z][lane] = s;
    __syncthreads();
    if (z == 0 && k < a.D) {
      double t = 0.0;
#pragma unroll
      for (int y = 0; y < 8; y += 2) t += red[y][lane] + red[y + 1][lane];
      a.G[(int64_t)c * a.ldq + k] = a.sign * (t + a.s2inv * q[k]);
    }
  }
  if (blockIdx.y == 0 && z == 1) {
    double lpv = 0.0, pr = 0.0;
    for (int ch = lane; ch < sp.chunks; ch += 64) lpv += Wlp[ch * stride + pos];
    for (int k = lane; k < a.D; k += 64) pr += q[k] * q[k];
    lpv = wave_sum(lpv);
    pr = wave_sum(pr);
    if (lane == 0) a.V[c] = -a.sign * (lpv - 0.5 * a.s2inv * pr);
  }
}

bool glm_wide_ok(int D) { return D > 128 && D <= 1024; }

GlmWidePlan glm_wide_plan(int C, int D, int num_cus, size_t max_doubles) {
  GlmWidePlan p;
  // 32 points per block feed each operand read to two products; 16 where that
  // holds every point, and above 512 columns (registers)
  p.gp = C > 16 && D <= 512 ? 32 : 16;
  const int groups = (C + p.gp - 1) / p.gp;
  int tb = num_cus > 0 ? num_cus : 256;
  if (tb < groups) tb = groups;
  // partials of any launch: one block's gp rows of D gradients, and gp log
  // densities, per block.  Where the gradient partials do not fit the
  // workspace the grid shrinks, down to one block per group, which writes G itself
  const size_t per = (size_t)p.gp * (D + 1);
  if (per * tb > max_doubles) {
    tb = (int)(max_doubles / per);
    if (tb < 2 * groups) {
      tb = groups;
      p.max_chunks = 1;
    }
  }
  p.total_blocks = tb;
  p.wg_doubles = p.max_chunks == 1 ? 0 : (size_t)tb * p.gp * D;
  p.work_doubles = p.wg_doubles + (size_t)tb * p.gp;
  return p;
}

template <int TW>
static void gw_launch(const GlmArgs& a, const GlmWidePlan& p, double* Wg, double* Wlp, hipStream_t st) {
  constexpr int W = 8;
  const dim3 grid(p.total_blocks), block(64 * W);
  if constexpr (TW <= 4) {
    if (p.gp == 32) {
      hipLaunchKernelGGL((glm_wide_f64<W, TW, 2>), grid, block, 0, st, a, p.total_blocks, p.max_chunks, Wg, Wlp);
      return;
    }
  }
  hipLaunchKernelGGL((glm_wide_f64<W, TW, 1>), grid, block, 0, st, a, p.total_blocks, p.max_chunks, Wg, Wlp);
}

int glm_grad_wide_f64(const GlmArgs& a, const GlmWidePlan& p, hipStream_t st) {
  if (!glm_wide_ok(a.D)) return 1;
  double* Wg = a.work;
  double* Wlp = a.work + p.wg_doubles;
  if (a.ev_begin) (void)hipEventRecord(a.ev_begin, st);
  // eight waves with as many 16-column tiles each as D needs
  switch ((a.D + 127) / 128) {
    case 2: gw_launch<2>(a, p, Wg, Wlp, st); break;
    case 3: gw_launch<3>(a, p, Wg, Wlp, st); break;
    case 4: gw_launch<4>(a, p, Wg, Wlp, st); break;
    case 5: gw_launch<5>(a, p, Wg, Wlp, st); break;
    case 6: gw_launch<6>(a, p, Wg, Wlp, st); break;
    case 7: gw_launch<7>(a, p, Wg, Wlp, st); break;
    default: gw_launch<8>(a, p, Wg, Wlp, st); break;
  }
  if (a.ev_end) (void)hipEventRecord(a.ev_end, st);
  hipLaunchKernelGGL(glm_wide_reduce, dim3(a.C, (a.D + 63) / 64), dim3(512), 0, st, a, p.total_blocks, p.max_chunks,
                     p.gp, Wg, Wlp);
  return 0;
}

}  // namespace nutsgpu
