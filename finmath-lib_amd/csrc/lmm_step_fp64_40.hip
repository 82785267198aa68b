// FP64 instantiations of the spot Euler path kernel for up to 40 forwards.
#include "lmm_spot.hpp"

namespace fm {
void launch_spot64_40(const StepArgs& a, hipStream_t stream) { launch_spot_n<5, double>(a, stream); }
}
