// FP32-mixed instantiations of the spot Euler path kernel up to 48 forwards, and the choice by size:
// capacities of 16, 32, 48 and 80 forwards in chunks of sixteen. The path arithmetic is in float, the
// numeraire and payoff/numeraire in double.
#include "lmm_spot.hpp"

namespace fm {
void launch_spot32_80(const StepArgs& a, hipStream_t stream);

// Pricing, simulation and the adjoint's forward pass (with checkpoints); a.Y0 holds the capped
// initial forwards.
void launch_lmm_step_fp32(const StepArgs& a, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (a.n <= 16) launch_spot_n<1, float>(a, s);
    else if (a.n <= 32) launch_spot_n<2, float>(a, s);
    else if (a.n <= 48) launch_spot_n<3, float>(a, s);
    else if (a.n <= 80) launch_spot32_80(a, s);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the path kernel");
}
}
