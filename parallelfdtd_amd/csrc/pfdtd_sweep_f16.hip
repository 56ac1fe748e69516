// pfdtd_sweep_f16.hip -- the several-level sweep's kernels for FP16 fields.
#include "pfdtd_sweep_kernel.h"

namespace pfdtd {

hipError_t launch_sweep_f16(const SweepPlan &p, const SweepArgsOf<h16> &a, int levels,
                           hipStream_t stream) {
  if (a.centred) return launch_any<h16, kCentred>(p, a, levels, stream);
  return launch_any<h16>(p, a, levels, stream);
}
hipError_t launch_sweep_diff(const SweepPlan &p, const SweepArgsOf<h16> &a, int levels,
                             hipStream_t stream) {
  return launch_any<h16, kDiff>(p, a, levels, stream);
}
hipError_t launch_pool_f16(int tiles, const void *args, const PoolJobDev *jobs, const PoolState *st,
                           const PoolLaunch &pl, int zc, int round, hipStream_t stream) {
  return launch_pool<h16>(tiles, args, jobs, st, pl, zc, round, stream);
}

}  // namespace pfdtd
