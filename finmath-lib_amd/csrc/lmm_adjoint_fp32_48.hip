// FP32-mixed instantiations of the reverse sweep for up to 48 forwards.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint32_48(const StepArgs& a, const AdjArgs& g, hipStream_t stream) { launch_spot_adjoint_n<3, float>(a, g, stream); }
}
