// FP32-mixed instantiations of the spot Euler path kernel: the path arithmetic in float (fused
// multiply-add allowed), numeraire and payoff/numeraire in double.
#include "lmm_spot.hpp"

namespace fm {
// pricing, simulation and the adjoint's forward pass: the spot kernel
void launch_lmm_step_fp32(const StepArgs& a, void* stream) {
    launch_spot<float>(a, (hipStream_t)stream);
}
}
