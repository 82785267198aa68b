// FP64 instantiations of the general path kernel: terminal or spot measure, carried or functional
// state. Compiled with -ffp-contract=off: the multiply-adds are written where they are meant.
#include "lmm_general64.hpp"

namespace fm {
void launch_lmm_step_general_fp64(const StepArgs& a, void* stream) { launch_general64<false, false>(a, (hipStream_t)stream); }
}
