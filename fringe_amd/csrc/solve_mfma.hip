// solve_mfma.hip -- launcher of the matrix-core estimator chain (mixed
// precisions, up to 32 dates).
#include <algorithm>

#include "solve_mfma.hpp"

namespace fringe {

void launch_solve_mfma(const SolveArgs& args, hipStream_t s) {
    SolveArgs a = args;
    long long pairs = (long long)a.n * (a.n - 1) / 2;
    if (a.module == FRINGE_MODULE_EVD && a.method == FRINGE_METHOD_STBAS) {
        pairs = 0;
        for (int i = 0; i < a.n; ++i) pairs += std::min(a.n, i + a.bw + 1) - i - 1;
    }
    a.inv_n = 1.0f / (float)a.n;
    a.inv_pairs = 1.0 / (double)pairs;
    a.inv_comp = 1.0 / (double)(a.n - a.ref);
    constexpr int WPB = 4;
    const dim3 grid((unsigned)((a.slots + WPB - 1) / WPB)), block(64 * WPB);
    if (a.module == FRINGE_MODULE_PHASE_LINK)
        hipLaunchKernelGGL((solve_mfma_kernel<MODE_EMI, WPB>), grid, block, 0, s, a);
    else if (a.method == FRINGE_METHOD_MLE)
        hipLaunchKernelGGL((solve_mfma_kernel<MODE_MLE, WPB>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((solve_mfma_kernel<MODE_EVD, WPB>), grid, block, 0, s, a);
}

}  // namespace fringe
