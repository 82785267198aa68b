// FP64 instantiations of the general path kernel with the predictor-corrector.
#include "lmm_general64.hpp"

namespace fm {
void launch_lmm_step_pc_fp64(const StepArgs& a, void* stream) { launch_general64<true, false>(a, (hipStream_t)stream); }
}
