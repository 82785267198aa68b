// FP64 instantiations of the reverse sweep up to 24 forwards, and the choice by size (the pricing
// pass's capacities). It recomputes the pricing pass's steps from its checkpointed states.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint64_40(const StepArgs& a, const AdjArgs& g, hipStream_t stream);
void launch_adjoint64_80(const StepArgs& a, const AdjArgs& g, hipStream_t stream);

void launch_lmm_adjoint_fp64(const StepArgs& a, const AdjArgs& g, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (a.n <= 8) launch_spot_adjoint_n<1, double>(a, g, s);
    else if (a.n <= 24) launch_spot_adjoint_n<3, double>(a, g, s);
    else if (a.n <= 40) launch_adjoint64_40(a, g, s);
    else if (a.n <= 80) launch_adjoint64_80(a, g, s);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the adjoint kernel");
}
}
