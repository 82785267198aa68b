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
    // blocks of paths by products and numeraires; a swap is one product per period, so there may be more of them
    // than the grid's second dimension holds
    const dim3 grid((unsigned)(((int64_t)a.P + kStepThreads - 1) / kStepThreads),
                    (unsigned)std::min<int64_t>((int64_t)a.num_products + a.n, 65535));
    hipLaunchKernelGGL(rows64_partials_kernel, grid, dim3(kStepThreads), 0, s, a);
    HIP_CHECK(hipGetLastError());
}
}
