// Batched gradient of the centered hierarchical logistic model (hier_logistic_cp)
// over many chains of one dataset.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace nutsgpu {

struct HlArgs {
  const double* block;   // device dataset block [N, K, G, mu_s, gstart[G+1], X, y]
  const double* Q;       // positions: row of the chain (idx or need) or of the position, stride ldq
  int64_t ldq;
  const int* idx;        // active positions -> chains; null: rows are positions
  const int* n_dev;      // active count (device) or null for n_rows
  // in place of idx, at most 64 chains: the chains' request flags (left as they
  // are); tally (optional) accumulates their number
  const int* need = nullptr;
  long long* tally = nullptr;
  int n_rows;
  double* Gout;          // gradient of V = -lp, stride ldg
  int64_t ldg;
  double* Vout;
  double* work;          // hl_work_doubles(G, K, n_rows)
  double jac;            // 1: add the log-Jacobian of tau = exp(v)
  double sign = 1.0;     // Gout, Vout as they are (V = -lp), or -1: log density and its gradient
};

void hl_grad_launch(const HlArgs& a, int G, int K, hipStream_t st);
size_t hl_work_doubles(int G, int K, int n_rows);

}  // namespace nutsgpu
