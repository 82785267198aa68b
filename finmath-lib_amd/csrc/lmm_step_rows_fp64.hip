// FP64 spot path kernel for few paths (lmm_rows64.hpp): capacities of 16, 32, 48 and 80 forwards. Compiled
// with -ffp-contract=off, as the kernel whose results it reproduces.
#include <algorithm>

#include "lmm_rows64.hpp"

namespace fm {
// a.values takes (num_slots + n + 1) * P doubles.
void launch_lmm_rows_fp64(const StepArgs& a, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    if (a.n <= 16) launch_rows64_n<1>(a, s);
    else if (a.n <= 32) launch_rows64_n<2>(a, s);
    else if (a.n <= 48) launch_rows64_n<3>(a, s);
    else if (a.n <= 80) launch_rows64_n<5>(a, s);
    else throw FmError(FM_ERR_UNSUPPORTED, "more than 80 forward rates are not supported by the path kernel");
    // products and numeraires by blocks of paths, in one grid dimension and rounds of at most a million: a swap is
    // one product per period, so there may be more than the 65,536 of the other dimensions
    const int64_t items = (((int64_t)a.P + kStepThreads - 1) / kStepThreads) * ((int64_t)a.num_products + a.n);
    const dim3 grid((unsigned)std::min<int64_t>(items, 1 << 20));
    hipLaunchKernelGGL(rows64_partials_kernel, grid, dim3(kStepThreads), 0, s, a);
    HIP_CHECK(hipGetLastError());
}
}
