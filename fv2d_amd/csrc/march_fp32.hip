// march_fp32.hip -- FP32-form instantiations of the register-march stage (U stored in FP32); those on
// the FP64 state are in march_fp32s64.hip.
#include "fv2d_march_device.h"

namespace fv2d {

hipError_t launch_march_fp32(const StageClass &c, const KParams &kp, const StageIO<float> &io, const MarchGeom &g,
                             const MarchCtl &mc, hipStream_t st) {
  return launch_march<float, float, DIVF_RUNTIME>(c, kp, io, g, mc, st);
}

}  // namespace fv2d
