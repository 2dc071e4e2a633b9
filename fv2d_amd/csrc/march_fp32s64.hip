// march_fp32s64.hip -- FP32-form instantiations of the register-march stage on a state stored in FP64
// (FV2D_FP32_STATE64).
#include "fv2d_march_device.h"

namespace fv2d {

hipError_t launch_march_fp32s64(const StageClass &c, const KParams &kp, const StageIO<double> &io, const MarchGeom &g,
                                const MarchCtl &mc, hipStream_t st) {
  return launch_march<float, double, DIVF_RUNTIME>(c, kp, io, g, mc, st);
}

}  // namespace fv2d
