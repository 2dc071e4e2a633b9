// march_fp64_exact.hip -- FP64 (parity form) register-march kernels for grids whose cell sizes
// are both powers of two (DIVF_EXACT). Built with -ffp-contract=off, as stage_fp64.hip.
#include "fv2d_march_device.h"

namespace fv2d {

hipError_t launch_march_fp64_exact(const StageClass &c, const KParams &kp, const StageIO<double> &io,
                                   const MarchGeom &g,
                             const MarchCtl &mc, hipStream_t st) {
  return launch_march<double, double, DIVF_EXACT>(c, kp, io, g, mc, st);
}

}  // namespace fv2d
