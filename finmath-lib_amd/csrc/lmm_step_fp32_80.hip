// FP32-mixed instantiations of the spot Euler path kernel for up to 80 forwards.
#include "lmm_spot.hpp"

namespace fm {
void launch_spot32_80(const StepArgs& a, hipStream_t stream) { launch_spot_n<5, float>(a, stream); }
}
