// pfdtd_sweep_f32.hip -- the several-level sweep's kernels for FP32 fields.
#include "pfdtd_sweep_kernel.h"

namespace pfdtd {

hipError_t launch_sweep_f32(const SweepPlan &p, const SweepArgsOf<float> &a, int levels,
                           hipStream_t stream) {
  if (a.centred) return launch_any<float, kCentred>(p, a, levels, stream);
  return launch_any<float>(p, a, levels, stream);
}
hipError_t launch_pool_f32(int tiles, const void *args, const PoolJobDev *jobs, const PoolState *st,
                           const PoolLaunch &pl, int zc, int round, hipStream_t stream) {
  return launch_pool<float>(tiles, args, jobs, st, pl, zc, round, stream);
}

}  // namespace pfdtd
