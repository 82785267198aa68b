// FP32-mixed instantiations of the reverse sweep.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_lmm_adjoint_fp32(const StepArgs& a, const AdjArgs& g, void* stream) { launch_spot_adjoint<float>(a, g, (hipStream_t)stream); }
}
