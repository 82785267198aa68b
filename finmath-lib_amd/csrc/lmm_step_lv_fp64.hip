// FP64 instantiations of the general path kernel with the local- and stochastic-volatility wrappers.
#include "lmm_general64.hpp"

namespace fm {
void launch_lmm_step_lvpc_fp64(const StepArgs& a, hipStream_t stream);

void launch_lmm_step_lv_fp64(const StepArgs& a, void* stream) {
    if (a.pc) launch_lmm_step_lvpc_fp64(a, (hipStream_t)stream);
    else launch_general64<false, true>(a, (hipStream_t)stream);
}
}
