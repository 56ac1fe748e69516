// pfdtd_sweep_f64.hip -- the several-level sweep's kernels for FP64 fields.
#include "pfdtd_sweep_kernel.h"

namespace pfdtd {

hipError_t launch_sweep_f64(const SweepPlan &p, const SweepArgsOf<double> &a, int levels,
                           hipStream_t stream) {
  if (a.centred) return launch_any<double, kCentred>(p, a, levels, stream);
  return launch_any<double>(p, a, levels, stream);
}

}  // namespace pfdtd
