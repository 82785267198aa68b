// FP64 instantiations of the reverse sweep: it recomputes the pricing pass's steps from its
// checkpointed states.
#include "lmm_spot_adjoint.hpp"

namespace fm {
void launch_lmm_adjoint_fp64(const StepArgs& a, const AdjArgs& g, void* stream) { launch_spot_adjoint<double>(a, g, (hipStream_t)stream); }
}
