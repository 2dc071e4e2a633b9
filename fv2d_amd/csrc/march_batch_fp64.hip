// march_batch_fp64.hip -- batched register-march kernels, FP64 form (same contraction flags as
// march_fp64.hip, so that a job's results are those of the single-simulation path bit for bit).
#include "fv2d_march_device.h"

namespace fv2d {

hipError_t launch_batch_march_fp64(const StageClass &c, const BatchJob *jobs, const BatchItem *items, const int *range,
                                   int *counter, int stage, int grid, hipStream_t st) {
  BatchMarchLaunch<double, double> f{jobs, items, range, counter, stage, grid, st};
  return with_class(c, f);
}

int batch_occupancy_march_fp64(const StageClass &c) {
  BatchMarchOcc<double, double> f;
  return with_class(c, f);
}

}  // namespace fv2d
