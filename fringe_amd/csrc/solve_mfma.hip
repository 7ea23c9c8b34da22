// solve_mfma.hip -- launcher of the matrix-core estimator chain (mixed
// precisions, up to 128 dates): one wave per pixel on a 16 x 16 tile up to 16
// dates and a 32 x 32 tile up to 32, one workgroup of a wave per 32 dates above.
#include "solve_mfma_wg.hpp"

namespace fringe {

template <int DIM> static void launch_wave(const SolveArgs& args, hipStream_t s) {
    constexpr int WPB = 4;
    slots_in_parts(args, 64, sizeof(cx<float>), [&](const SolveArgs& a) {
        const dim3 grid((unsigned)((a.slots + WPB - 1) / WPB)), block(64 * WPB);
        if (a.module == FRINGE_MODULE_PHASE_LINK)
            hipLaunchKernelGGL((solve_mfma_kernel<MODE_EMI, DIM, WPB>), grid, block, 0, s, a);
        else if (a.method == FRINGE_METHOD_MLE)
            hipLaunchKernelGGL((solve_mfma_kernel<MODE_MLE, DIM, WPB>), grid, block, 0, s, a);
        else
            hipLaunchKernelGGL((solve_mfma_kernel<MODE_EVD, DIM, WPB>), grid, block, 0, s, a);
    });
}

template <int NT> static void launch_wg(const SolveArgs& args, hipStream_t s) {
    slots_in_parts(args, 64 * NT, sizeof(cx<float>), [&](const SolveArgs& a) {
        const dim3 grid((unsigned)a.slots), block(64 * NT);
        if (a.module == FRINGE_MODULE_PHASE_LINK)
            hipLaunchKernelGGL((solve_mfma_wg_kernel<MODE_EMI, NT>), grid, block, 0, s, a);
        else if (a.method == FRINGE_METHOD_MLE)
            hipLaunchKernelGGL((solve_mfma_wg_kernel<MODE_MLE, NT>), grid, block, 0, s, a);
        else
            hipLaunchKernelGGL((solve_mfma_wg_kernel<MODE_EVD, NT>), grid, block, 0, s, a);
    });
}

void launch_solve_mfma(const SolveArgs& args, bool bf16, hipStream_t s) {
    SolveArgs a = args;
    set_solve_counts(a);
    const float n = (float)a.n;
    a.cert_h = 5.9604645e-8f * (bf16 ? kCertScale : fminf(kCertScaleH, kCertScaleH * 48.0f / n));
    a.cert_g = 5.9604645e-8f * (bf16 ? kCertScale : fminf(kCertScale, fmaxf(kCertScaleG, kCertScale * 8.0f / n)));
    if (a.n > 96) launch_wg<4>(a, s);
    else if (a.n > 64) launch_wg<3>(a, s);
    else if (a.n > 32) launch_wg<2>(a, s);
    else if (a.n > 16) launch_wave<32>(a, s);
    else launch_wave<16>(a, s);
}

}  // namespace fringe
