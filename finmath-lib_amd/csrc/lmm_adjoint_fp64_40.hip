// FP64 instantiations of the reverse sweep for up to 40 forwards.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_adjoint64_40(const StepArgs& a, const AdjArgs& g, hipStream_t stream) { launch_spot_adjoint_n<5, double>(a, g, stream); }
}
