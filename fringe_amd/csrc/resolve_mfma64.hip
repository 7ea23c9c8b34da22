// resolve_mfma64.hip -- launches of the FP64 re-solve of the pixels the mixed
// precisions did not certify (up to 128 dates), on the plain FP64 path's
// estimator chain.
#include <algorithm>

#include "engine_internal.hpp"
#include "solve_mfma64.hpp"

namespace fringe {

// The Gram's position list, then the chain's share of the inverse.
template <int NW> static size_t scratch(int Nx, int Ny) {
    return std::max(gram_list_bytes(Nx, Ny), keep64_bytes<MODE_EMI, NW>());
}

template <int NW> static void launch(const SolveArgs& a, unsigned blocks, hipStream_t s) {
    const dim3 grid(blocks), block(64 * NW);
    const size_t lds = scratch<NW>(a.g64.Nx, a.g64.Ny);
    if (a.module == FRINGE_MODULE_PHASE_LINK)
        hipLaunchKernelGGL((resolve_mfma64_kernel<MODE_EMI, NW>), grid, block, lds, s, a);
    else if (a.method == FRINGE_METHOD_MLE)
        hipLaunchKernelGGL((resolve_mfma64_kernel<MODE_MLE, NW>), grid, block, lds, s, a);
    else
        hipLaunchKernelGGL((resolve_mfma64_kernel<MODE_EVD, NW>), grid, block, lds, s, a);
}

void launch_resolve_mfma64(const SolveArgs& args, unsigned blocks, hipStream_t s) {
    SolveArgs a = args;
    set_solve_counts(a);
    switch ((a.n + 15) / 16) {
        case 1: launch<1>(a, blocks, s); break;
        case 2: launch<2>(a, blocks, s); break;
        case 3: launch<3>(a, blocks, s); break;
        case 4: launch<4>(a, blocks, s); break;
        case 5: launch<5>(a, blocks, s); break;
        case 6: launch<6>(a, blocks, s); break;
        case 7: launch<7>(a, blocks, s); break;
        default: launch<8>(a, blocks, s); break;
    }
}

}  // namespace fringe
