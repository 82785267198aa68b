// FP64 instantiations of the spot Euler path kernel for up to 80 forwards.
#include "lmm_spot64.hpp"

namespace fm {
void launch_spot64_80(const StepArgs& a, hipStream_t stream) { launch_spot64_n<10>(a, stream); }
}
