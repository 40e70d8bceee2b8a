// Batched FP64 logistic-regression gradient for more coefficients than the
// single-wave kernels hold (128 < D <= 1024).
#pragma once
#include "launch.h"

namespace nutsgpu {

struct GlmWidePlan {
  int max_chunks = 1 << 30; // 1: the workspace has no room for gradient partials
  int total_blocks = 0;     // grid of every launch (the split adapts to the active count)
  int gp = 16;              // points per block
  size_t wg_doubles = 0;    // gradient partials (0: one chunk, written to G directly)
  size_t work_doubles = 0;  // with the log-density partials
};

bool glm_wide_ok(int D);
// max_doubles bounds the workspace of the gradient partials
GlmWidePlan glm_wide_plan(int C, int D, int num_cus, size_t max_doubles = (size_t)1 << 40);
int glm_grad_wide_f64(const GlmArgs& a, const GlmWidePlan& p, hipStream_t st);

}  // namespace nutsgpu
