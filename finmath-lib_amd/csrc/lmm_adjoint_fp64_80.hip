// FP64 instantiations of the reverse sweep for up to 80 forwards.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint64_80(const StepArgs& a, const AdjArgs& g, hipStream_t stream) { launch_spot_adjoint_n<10, double>(a, g, stream); }
}
