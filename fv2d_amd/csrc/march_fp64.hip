// march_fp64.hip -- FP64 (parity form) instantiations of the register-march stage with the
// general division form; the exact-division ones are in march_fp64_exact.hip. Built with
// -ffp-contract=off, as stage_fp64.hip.
#include "fv2d_march_device.h"

namespace fv2d {

hipError_t launch_march_fp64(const StageClass &c, const KParams &kp, const StageIO<double> &io, const MarchGeom &g,
                             const MarchCtl &mc, hipStream_t st) {
  if (kp.divx == DIV_EXACT && kp.divy == DIV_EXACT) return launch_march_fp64_exact(c, kp, io, g, mc, st);
  return launch_march<double, double, DIVF_GENERAL>(c, kp, io, g, mc, st);
}

}  // namespace fv2d
