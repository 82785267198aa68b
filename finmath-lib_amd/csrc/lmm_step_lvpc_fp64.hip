// FP64 instantiations of the general path kernel with the wrappers and the predictor-corrector.
#include "lmm_general64.hpp"

namespace fm {
void launch_lmm_step_lvpc_fp64(const StepArgs& a, hipStream_t stream) { launch_general64<true, true>(a, stream); }
}
