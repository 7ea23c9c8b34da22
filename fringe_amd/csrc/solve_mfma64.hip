// solve_mfma64.hip -- launches of the plain FP64 path on the matrix cores (up
// to 128 dates): the coherence of a range of slots, and the estimator chain.
#include "solve_mfma64.hpp"

namespace fringe {

template <int NW> static void launch(const SolveArgs& args, hipStream_t s) {
    slots_in_parts(args, 64 * NW, sizeof(cx<double>), [&](const SolveArgs& a) {
        const dim3 grid((unsigned)a.slots), block(64 * NW);
        if (a.module == FRINGE_MODULE_PHASE_LINK)
            hipLaunchKernelGGL((solve_mfma64_kernel<MODE_EMI, NW>), grid, block, (keep64_bytes<MODE_EMI, NW>()), s, a);
        else if (a.method == FRINGE_METHOD_MLE)
            hipLaunchKernelGGL((solve_mfma64_kernel<MODE_MLE, NW>), grid, block, (keep64_bytes<MODE_MLE, NW>()), s, a);
        else
            hipLaunchKernelGGL((solve_mfma64_kernel<MODE_EVD, NW>), grid, block, (keep64_bytes<MODE_EVD, NW>()), s, a);
    });
}

void launch_solve_mfma64(const SolveArgs& args, hipStream_t s) {
    SolveArgs a = args;
    set_solve_counts(a);
    switch ((a.n + 15) / 16) {   // one wave per 16 dates
        case 1: launch<1>(a, s); break;
        case 2: launch<2>(a, s); break;
        case 3: launch<3>(a, s); break;
        case 4: launch<4>(a, s); break;
        case 5: launch<5>(a, s); break;
        case 6: launch<6>(a, s); break;
        case 7: launch<7>(a, s); break;
        default: launch<8>(a, s); break;
    }
}

template <int NW> static void launch_gram(const GramArgs& args, hipStream_t s) {
    slots_in_parts(args, 64 * NW, sizeof(cx<double>), [&](const GramArgs& a) {
        hipLaunchKernelGGL((gram_mfma64_kernel<NW>), dim3((unsigned)a.slots), dim3(64 * NW), gram_list_bytes(a.Nx, a.Ny), s,
                           a);
    });
}

void launch_gram_mfma64(const GramArgs& a, hipStream_t s) {
    switch ((a.n + 15) / 16) {
        case 1: launch_gram<1>(a, s); break;
        case 2: launch_gram<2>(a, s); break;
        case 3: launch_gram<3>(a, s); break;
        case 4: launch_gram<4>(a, s); break;
        case 5: launch_gram<5>(a, s); break;
        case 6: launch_gram<6>(a, s); break;
        case 7: launch_gram<7>(a, s); break;
        default: launch_gram<8>(a, s); break;
    }
}

}  // namespace fringe
