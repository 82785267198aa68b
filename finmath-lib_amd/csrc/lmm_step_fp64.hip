// FP64 instantiations of the spot Euler path kernel up to 24 forwards, and the choice by size:
// capacities of 8, 24, 40 and 80 forwards in chunks of eight. Compiled with -ffp-contract=off: the
// multiply-adds are written where they are meant. The larger capacities are translation units of
// their own, which compile side by side.
#include "lmm_spot.hpp"

namespace fm {
void launch_spot64_40(const StepArgs& a, hipStream_t stream);
void launch_spot64_80(const StepArgs& a, hipStream_t stream);

// Pricing, simulation and the adjoint's forward pass (with checkpoints); a.Y0 holds the initial states.
void launch_lmm_step_fp64(const StepArgs& a, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (a.n <= 8) launch_spot_n<1, double>(a, s);
    else if (a.n <= 24) launch_spot_n<3, double>(a, s);
    else if (a.n <= 40) launch_spot64_40(a, s);
    else if (a.n <= 80) launch_spot64_80(a, s);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the path kernel");
}
}
