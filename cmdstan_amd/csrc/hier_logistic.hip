// Batched gradient of the centered hierarchical logistic model for many chains
// (one dataset):
//   mu_k ~ N(0, mu_s), tau_k = exp(v_k) ~ HalfNormal(1) (+ v_k Jacobian),
//   beta[g][k] ~ N(mu_k, tau_k), y_n ~ bernoulli_logit(x_n . beta[group_n]).
// Kernel 1 takes one group and a tile of points per block: a lane owns one point
// and keeps its beta[g] and gradient in registers (K <= 16, a template parameter:
// the K products of an observation are straight-line code on broadcast LDS reads),
// and the block's other lanes split the observations -- four ways for a tile of
// 64 points (one wave each), sixteen ways for a tile of 16, where most lanes of a
// 64-point tile would have no point.  It writes the beta[g] gradient directly and
// per-group partials for the hyperparameters; kernel 2 reduces those over groups
// in a fixed order (deterministic, no atomics).
// Bound: the FP64 vector unit (4 K + some 45 operations per observation and
// point).  log(1 + e^eta) is a factor of one product per lane, its logarithm
// taken once at the end (LogProduct).
// Dataset block (host layout): [N, K, G, mu_s, gstart[G+1], X[N*K] sorted by group, y[N]].
#include "device_common.h"
#include "hier_logistic.h"

namespace nutsgpu {

#define HL_OBS 128   // observations staged per LDS pass
#define HL_HW 16     // waves of a hyperparameter block

// partials of the hyperparameters: column j of group g at ((j G) + g) n + pos
// (j < K d lp / d mu_k, then d lp / d tau_k, last the log density), so the lanes of
// a tile store runs of points and kernel 2 reads them back as such
template <int K, int TC>
__global__ void __launch_bounds__(256) hl_group_kernel(HlArgs a) {
  constexpr int SPLIT = 256 / TC;  // observations split this many ways
  __shared__ double sX[HL_OBS * K];
  __shared__ double sY[HL_OBS];
  __shared__ double sRed[SPLIT][TC][K + 1];
  __shared__ int sRow[TC];  // rows of the tile's points
  const double* d = a.block;
  const int G = (int)d[2];
  const double* gstart = d + 4;
  const double* X = d + 5 + G;
  const int N = (int)d[0];
  const double* y = X + (int64_t)N * K;
  const int g = blockIdx.x % G;
  const int tile = blockIdx.x / G;
  const ActiveChains act(a.need, a.idx, a.n_dev, a.n_rows);
  const int n_act = min(a.n_rows, act.n);
  const int p0 = tile * TC;
  if (p0 >= n_act) return;
  const int t = threadIdx.x, w = t / TC, lane = t % TC;
  const int pos = p0 + lane;
  const bool live = pos < n_act;
  const int64_t row = act.at(pos);
  if (t < TC) sRow[t] = (int)row;
  const double* q = a.Q + row * a.ldq;
  double b[K], gb[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    b[k] = live ? q[2 * K + (int64_t)g * K + k] : 0.0;
    gb[k] = 0.0;
  }
  double lp = 0.0;
  LogProduct lg;
  const int n0 = (int)gstart[g], n1 = (int)gstart[g + 1];
  for (int base = n0; base < n1; base += HL_OBS) {
    const int cnt = min(HL_OBS, n1 - base);
    __syncthreads();
    for (int i = t; i < cnt * K; i += 256) sX[i] = X[(int64_t)base * K + i];
    for (int i = t; i < cnt; i += 256) sY[i] = y[base + i];
    __syncthreads();
    // two observations per step: independent exponentials in flight
    for (int n = w; n < cnt; n += 2 * SPLIT) {
      const int n2 = n + SPLIT;
      const bool two = n2 < cnt;
      const double* xr = sX + n * K;
      const double* xr2 = sX + (two ? n2 : n) * K;
      double x1[K], x2[K], e = 0.0, e2 = 0.0;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        x1[k] = xr[k];
        x2[k] = xr2[k];
        e += x1[k] * b[k];
        e2 += x2[k] * b[k];
      }
      const double yy = sY[n], yy2 = two ? sY[n2] : 0.0;
      const double t1 = exp(-fabs(e)), t2 = exp(-fabs(e2));
      const double d1 = 1.0 + t1, d2 = 1.0 + t2;
      const double r = yy - (e >= 0.0 ? 1.0 : t1) * recip_small(d1);
      const double s2 = yy2 - (e2 >= 0.0 ? 1.0 : t2) * recip_small(d2);
      const double r2 = two ? s2 : 0.0;
      lp += yy * e - (e > 0.0 ? e : 0.0);
      lg.times(t1, d1);
      if (two) {
        lp += yy2 * e2 - (e2 > 0.0 ? e2 : 0.0);
        lg.times(t2, d2);
      }
#pragma unroll
      for (int k = 0; k < K; ++k) gb[k] += r * x1[k] + r2 * x2[k];
    }
    lg.fold();  // at most HL_OBS / SPLIT factors since the last
  }
  // combine the partial sums of the observation split
#pragma unroll
  for (int k = 0; k < K; ++k) sRed[w][lane][k] = gb[k];
  sRed[w][lane][K] = lp - lg.log_value();
  __syncthreads();
  // thread (point, k): beta gradient and the hyperparameters' partials
  for (int i = t; i < TC * K; i += 256) {
    const int ln = i % TC, k = i / TC;
    const int ps = p0 + ln;
    if (ps >= n_act) continue;
    const int64_t ro = sRow[ln];
    const double* qp = a.Q + ro * a.ldq;
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < SPLIT; ++ww) s += sRed[ww][ln][k];
    const double mu = qp[k], v = qp[K + k], bk = qp[2 * K + (int64_t)g * K + k];
    const double it = exp(-v);  // 1 / tau
    const double dd = bk - mu;
    const double z = dd * it;
    const double dz = z * it;  // (beta - mu) / tau^2
    // d lp / d beta = likelihood score - (beta - mu) / tau^2
    a.Gout[ro * a.ldg + 2 * K + (int64_t)g * K + k] = a.sign * (dz - s);
    a.work[((int64_t)k * G + g) * a.n_rows + ps] = dz;                   // d/d mu
    a.work[((int64_t)(K + k) * G + g) * a.n_rows + ps] = z * dz - it;    // d/d tau
    if (k == 0) {
      double lpt = 0.0;
#pragma unroll
      for (int ww = 0; ww < SPLIT; ++ww) lpt += sRed[ww][ln][K];
#pragma unroll
      for (int kk = 0; kk < K; ++kk) {
        const double vk = qp[K + kk];
        const double zk = (qp[2 * K + (int64_t)g * K + kk] - qp[kk]) * exp(-vk);
        lpt += -vk - 0.5 * zk * zk;
      }
      a.work[((int64_t)(2 * K) * G + g) * a.n_rows + ps] = lpt;
    }
  }
}

// hyperparameters: a block per (column of the partials, 64 points), sixteen
// waves over the groups (lane = point, so every read is a run of points), then
// one thread per point; the log density's column also takes the priors.  A wave
// is a chain of G / (8 HL_HW) waits for memory: with four waves 9.7 us at 256
// points and 400 groups, now 7.3 us (50 groups, 64 points: 5.3, 4.8)
__global__ void __launch_bounds__(64 * HL_HW) hl_hyper_kernel(HlArgs a) {
  __shared__ double red[HL_HW][64];
  const double* d = a.block;
  const int K = (int)d[1], G = (int)d[2];
  const double mu_s = d[3];
  const ActiveChains act(a.need, a.idx, a.n_dev, a.n_rows);
  const int n_act = min(a.n_rows, act.n);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int p0 = blockIdx.x * 64, j = blockIdx.y;
  if (p0 >= n_act) return;
  if (a.tally && p0 == 0 && j == 0 && threadIdx.x == 0) *a.tally += n_act;
  const int pos = p0 + lane;
  const int64_t row = act.at(pos);
  double s = 0.0;
  if (pos < n_act) {
    const double* col = a.work + (int64_t)j * G * a.n_rows + pos;
#pragma unroll 8
    for (int g = w; g < G; g += HL_HW) s += col[(int64_t)g * a.n_rows];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w != 0 || pos >= n_act) return;
  s = 0.0;
#pragma unroll
  for (int v = 0; v < HL_HW; v += 2) s += red[v][lane] + red[v + 1][lane];
  const double* q = a.Q + row * a.ldq;
  double* gout = a.Gout + row * a.ldg;
  if (j < K) {
    gout[j] = a.sign * (q[j] / (mu_s * mu_s) - s);
  } else if (j < 2 * K) {
    const double tau = exp(q[j]);
    gout[j] = -a.sign * (a.jac + tau * (s - tau));
  } else {
    double lp = s;
    for (int k = 0; k < K; ++k) {
      const double mu = q[k], v = q[K + k], tau = exp(v);
      lp += -0.5 * mu * mu / (mu_s * mu_s) - 0.5 * tau * tau + a.jac * v;
    }
    a.Vout[row] = -a.sign * lp;
  }
}

template <int K>
static void hl_group_launch(const HlArgs& a, int G, hipStream_t st) {
  // tiles of 16 points while a 64-point tile would be less than half full
  if (a.n_rows <= 32)
    hipLaunchKernelGGL((hl_group_kernel<K, 16>), dim3(G * ((a.n_rows + 15) / 16)), dim3(256), 0, st, a);
  else hipLaunchKernelGGL((hl_group_kernel<K, 64>), dim3(G * ((a.n_rows + 63) / 64)), dim3(256), 0, st, a);
}

void hl_grad_launch(const HlArgs& a, int G, int K, hipStream_t st) {
  switch (K) {
#define HL_CASE(k) case k: hl_group_launch<k>(a, G, st); break;
    HL_CASE(1) HL_CASE(2) HL_CASE(3) HL_CASE(4) HL_CASE(5) HL_CASE(6) HL_CASE(7) HL_CASE(8)
    HL_CASE(9) HL_CASE(10) HL_CASE(11) HL_CASE(12) HL_CASE(13) HL_CASE(14) HL_CASE(15) HL_CASE(16)
#undef HL_CASE
    default: return;  // the model is refused at K > 16
  }
  hipLaunchKernelGGL(hl_hyper_kernel, dim3((a.n_rows + 63) / 64, 2 * K + 1), dim3(64 * HL_HW), 0, st, a);
}

size_t hl_work_doubles(int G, int K, int n_rows) { return (size_t)G * n_rows * (2 * K + 1); }

}  // namespace nutsgpu
