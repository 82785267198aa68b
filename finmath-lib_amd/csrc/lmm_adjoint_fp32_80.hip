// FP32-mixed instantiations of the reverse sweep for up to 80 forwards.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint32_80(const StepArgs& a, const AdjArgs& g, hipStream_t stream) { launch_spot_adjoint_n<5, float>(a, g, stream); }
}
