// The fused NUTS state machine for chains whose vectors fit LDS (one wave per
// block and chain).  Compiled with -ffp-contract=off like nuts_kernels.hip.
#include "launch.h"
#include "models_device.h"
#include "nuts_device.h"

namespace nutsgpu {

template <int METRIC, class F, class VT>
__global__ void __launch_bounds__(NUTS_WAVE) advance_fused_lds_kernel(NutsParams P, NutsBuffers B, F f) {
  nuts_advance_lds_body<METRIC, F, VT>(P, B, f);
}

// LDS bytes of a chain's vectors, or 0 where the global-memory machine runs: a
// chain's vectors have to fit one block's LDS, and every chain to be resident
// at once (a second round of blocks would wait for the first's whole launch;
// two waves per SIMD is what the machine's registers allow, eight chains a CU).
static size_t fused_lds_bytes(int metric, bool vec32, const NutsParams& P, const NutsBuffers& B) {
  struct Limits { size_t lds; int cus; };
  static const Limits lim = [] {
    int dev = 0, lds = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return Limits{0, 0};
    return Limits{(size_t)lds, cus};
  }();
  const size_t fixed = sizeof(ChainState) + (metric == METRIC_DENSE ? NUTS_WAVE * DENSE_RMAX * sizeof(double) : 0) + 256;
  const size_t bytes = nuts_lds_vector_bytes(B.max_Dp, P.NV, vec32 ? sizeof(float) : sizeof(double));
  if (bytes + fixed > lim.lds) return 0;
  const int per_cu = (int)(lim.lds / (bytes + fixed));
  return (int64_t)B.C <= (int64_t)lim.cus * (per_cu < 8 ? per_cu : 8) ? bytes : 0;
}

template <class F>
static void lds_for_metric(int metric, bool vec32, size_t lds, const NutsParams& P, const NutsBuffers& B, const F& f,
                           hipStream_t st) {
  const dim3 grid(B.C), blk(NUTS_WAVE);
  if constexpr (F::vec32) {
    if (vec32) {
      if (metric == METRIC_UNIT)
        hipLaunchKernelGGL((advance_fused_lds_kernel<METRIC_UNIT, F, float>), grid, blk, lds, st, P, B, f);
      else hipLaunchKernelGGL((advance_fused_lds_kernel<METRIC_DIAG, F, float>), grid, blk, lds, st, P, B, f);
      return;
    }
  }
  if (metric == METRIC_UNIT)
    hipLaunchKernelGGL((advance_fused_lds_kernel<METRIC_UNIT, F, double>), grid, blk, lds, st, P, B, f);
  else if (metric == METRIC_DENSE)
    hipLaunchKernelGGL((advance_fused_lds_kernel<METRIC_DENSE, F, double>), grid, blk, lds, st, P, B, f);
  else hipLaunchKernelGGL((advance_fused_lds_kernel<METRIC_DIAG, F, double>), grid, blk, lds, st, P, B, f);
}

bool launch_advance_fused_lds(int kind, int metric, bool vec32, const NutsParams& P, const NutsBuffers& B,
                              const ModelDataDev& md, hipStream_t st) {
  const size_t lds = fused_lds_bytes(metric, vec32, P, B);
  if (lds == 0) return false;
  NUTS_MODEL_SWITCH(kind, md, lds_for_metric(metric, vec32, lds, P, B, f, st));
  return true;
}

}  // namespace nutsgpu
