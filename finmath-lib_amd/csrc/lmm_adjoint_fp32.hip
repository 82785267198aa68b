// FP32-mixed instantiations of the reverse sweep up to 32 forwards, and the choice by size (the pricing
// pass's capacities).
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint32_48(const StepArgs& a, const AdjArgs& g, hipStream_t stream);
void launch_adjoint32_80(const StepArgs& a, const AdjArgs& g, hipStream_t stream);

void launch_lmm_adjoint_fp32(const StepArgs& a, const AdjArgs& g, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (a.n <= 16) launch_spot_adjoint_n<1, float>(a, g, s);
    else if (a.n <= 32) launch_spot_adjoint_n<2, float>(a, g, s);
    else if (a.n <= 48) launch_adjoint32_48(a, g, s);
    else if (a.n <= 80) launch_adjoint32_80(a, g, s);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the adjoint kernel");
}
}
