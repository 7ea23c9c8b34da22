// solvers.hip -- which estimator chain serves a launch, and the launches of
// the vector-unit chains (one row per lane at 33-64 dates, a work matrix
// above 64): single grids, persistent queues, the FP64 re-solve of a tile's
// pixel list.  Up to 128 dates the matrix-core chains (solve_mfma.hip,
// solve_mfma64.hip) serve every launch unless the schedule asks for another.
#include <algorithm>

#include "device_common.hpp"
#include "engine_internal.hpp"
#include "link_solve.hpp"
#include "solve32.hpp"
#include "timing.hpp"

namespace fringe {

// Above 64 dates: one pixel per two-wave workgroup, rows g + 128 q; the
// work matrix in LDS, or at a.awork when it does not fit there.
template <typename T, typename Tg, int R>
static void launch_solve_generic(SolveArgs a, hipStream_t s) {
    a.group_bytes = solve_group_bytes<T>(a.n, a.awork == nullptr);
    hipLaunchKernelGGL((solve_kernel<T, Tg, 128, R, false>), dim3((unsigned)a.slots), dim3(128), a.group_bytes, s,
                       a);
}

// The matrix-core chains (FP32 in the mixed precisions, FP64 in the plain
// path and the re-solve) serve every launch up to 32 dates, and 33..128 dates
// where the schedule FRINGE_SCHED_GENERIC_A (or its default) asks for rows in
// registers.
bool matrix_solver_selected(int n, int precision) {
    if (n <= 32) return true;
    if (n > kMaxBandsMfma) return false;
    const int pk = precision == FRINGE_PREC_FP64 ? 0 : 1;
    // FP32 at 49..64 dates: 0 is the default's value, and the matrix cores too
    // (one row per lane took 15.1 ms for 131 k pixels of 64 dates, they 3.9)
    if (pk == 1 && n > 48 && n <= 64) return true;
    return schedule_lookup(FRINGE_SCHED_GENERIC_A, n, pk, 0, generic_a_default(n, pk)) == 2;
}

// 32 < n <= 64: one row per lane, one pixel per wave.
template <typename T, typename Tg> static void launch_lanes(const SolveArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)a.slots), block(64);
    if (a.module == FRINGE_MODULE_PHASE_LINK)
        hipLaunchKernelGGL((solve_reg_kernel<T, Tg, MODE_EMI, 64, false>), grid, block, 0, s, a);
    else if (a.method == FRINGE_METHOD_MLE)
        hipLaunchKernelGGL((solve_reg_kernel<T, Tg, MODE_MLE, 64, false>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((solve_reg_kernel<T, Tg, MODE_EVD, 64, false>), grid, block, 0, s, a);
}

// 64 < n <= 256: a work matrix in LDS, or at a.awork.
template <typename T, typename Tg> static void launch_work(const SolveArgs& a, hipStream_t s) {
    if (a.n <= 128) launch_solve_generic<T, Tg, 1>(a, s);
    else launch_solve_generic<T, Tg, 2>(a, s);
}

void launch_solve(const SolveArgs& a, int precision, hipStream_t s) {
    const bool fp64 = precision == FRINGE_PREC_FP64;
    if (matrix_solver_selected(a.n, precision)) {
        if (fp64) launch_solve_mfma64(a, s);
        else launch_solve_mfma(a, precision == FRINGE_PREC_MIXED_BF16, s);
    } else if (a.n <= 64) {
        if (fp64) launch_lanes<double, double>(a, s);
        else launch_lanes<float, float>(a, s);
    } else if (fp64) {
        launch_work<double, double>(a, s);
    } else if (link_uses_mfma(a.n, precision)) {
        launch_work<float, float>(a, s);   // the MFMA Gram's complex64 coherence
    } else {
        launch_work<float, double>(a, s);
    }
}

// Static LDS of the solver kernels that run above 64 dates (their reduction
// scratch); the launch checks add it to the dynamic LDS of a pixel.
size_t solve_static_lds(int precision) {
    hipFuncAttributes fa{};
    size_t most = 0;
    const void* ks[2] = {precision == FRINGE_PREC_FP64 ? (const void*)solve_kernel<double, double, 128, 2, false>
                                                        : (const void*)solve_kernel<float, double, 128, 2, false>,
                         precision == FRINGE_PREC_FP64 ? (const void*)solve_kernel<double, double, 128, 1, false>
                                                        : (const void*)solve_kernel<float, float, 128, 1, false>};
    for (const void* k : ks) most = std::max<size_t>(most, hipFuncGetAttributes(&fa, k) == hipSuccess
                                                               ? fa.sharedSizeBytes : 256);
    return most;
}

// Whether the work matrix of the solver above 64 dates fits in LDS.
// The schedule FRINGE_SCHED_GENERIC_A may move it to global memory even
// when it fits: the pixels in flight are then limited by registers, not LDS.
bool solve_a_in_lds(int n, int precision) {
    if (matrix_solver_selected(n, precision)) return true;   // no work matrix at all
    if (schedule_lookup(FRINGE_SCHED_GENERIC_A, n, precision == FRINGE_PREC_FP64 ? 0 : 1, 0, 0) == 1) return false;
    const size_t b = precision == FRINGE_PREC_FP64 ? solve_group_bytes<double>(n) : solve_group_bytes<float>(n);
    return b + solve_static_lds(precision) <= (size_t)device_lds_limit();
}

// Per-workgroup global area of the FP64 re-solve above 64 dates: the FP64
// coherence, then the work matrix.
size_t resolve_generic_area_bytes(int n) {
    const int S = n | 1;
    return align256((size_t)n * n * sizeof(cx<double>)) + align256((size_t)n * S * sizeof(cx<double>));
}

size_t resolve_generic_lds_bytes(int n, int Nx, int Ny) {
    return solve_group_bytes<double>(n, false) + 2 * gram_f64_group_bytes(n, Nx, Ny, kResolveCB) +
           solve_static_lds(FRINGE_PREC_FP64);
}

// FP64 re-solve (Gram and estimator chain of the plain FP64 path) of the
// pixels the FP32 solver of this tile listed as not certified.  Each
// workgroup loops over its share of the list with its pixel's coherence
// (and, above 64 dates, work matrix) in its own area at P.d_rwork.
static void launch_resolve(const LinkPlan& P, const uint32_t* wts, SolveArgs a, hipStream_t s) {
    GramArgs g{};
    g.slc = a.slc;
    g.wts = wts;
    g.rows = P.rows;
    g.cols = P.cols;
    g.n = P.n;
    g.Nx = P.Nx;
    g.Ny = P.Ny;
    g.nul = P.nul;
    g.min_nb = P.min_nb;
    g.npx = P.npx;
    a.g64 = g;
    a.list = P.d_cert_list;
    a.list_count = P.d_cert_count;
    a.list_cap = P.cert_cap;
    a.awork = P.d_rwork;
    a.awork_stride = P.n <= 64 ? resolve_small_area_bytes(P.n) : resolve_generic_area_bytes(P.n);
    const int areas = P.resolve_areas ? P.resolve_areas
                      : P.n <= 64     ? resolve_small_areas(P.n, kResolveAreaBudget)
                                      : resolve_generic_blocks(a.awork_stride);
    if (matrix_solver_selected(P.n, FRINGE_PREC_FP64)) {
        launch_resolve_mfma64(a, (unsigned)areas, s);
        return;
    }
    const dim3 grid((unsigned)areas);
    if (P.n <= 64) {
        a.group_bytes = resolve_group_bytes(P.n, P.Nx, P.Ny);
        const size_t lds = a.group_bytes;
        if (a.module == FRINGE_MODULE_PHASE_LINK)
            hipLaunchKernelGGL((solve_reg_kernel<double, double, MODE_EMI, 64, true>), grid, dim3(64), lds, s, a);
        else if (a.method == FRINGE_METHOD_MLE)
            hipLaunchKernelGGL((solve_reg_kernel<double, double, MODE_MLE, 64, true>), grid, dim3(64), lds, s, a);
        else
            hipLaunchKernelGGL((solve_reg_kernel<double, double, MODE_EVD, 64, true>), grid, dim3(64), lds, s, a);
        return;
    }
    a.group_bytes = solve_group_bytes<double>(P.n, false);
    const size_t lds = a.group_bytes + 2 * gram_f64_group_bytes(P.n, P.Nx, P.Ny, kResolveCB);
    if (P.n <= 128)
        hipLaunchKernelGGL((solve_kernel<double, double, 128, 1, true>), grid, dim3(128), lds, s, a);
    else
        hipLaunchKernelGGL((solve_kernel<double, double, 128, 2, true>), grid, dim3(128), lds, s, a);
}

// LDS of one lane group of the re-solve up to 64 dates: the Gram's scratch.
size_t resolve_group_bytes(int n, int Nx, int Ny) { return gram_f64_group_bytes(n, Nx, Ny, kResolveSmallCB); }

size_t resolve_small_area_bytes(int n) { return align256((size_t)n * n * sizeof(cx<double>)); }

int resolve_small_areas(int n, size_t budget) {
    const size_t most = n <= 32 ? 2048 : 1024, least = n <= 32 ? 32 : 16;
    const size_t k = (budget / 4) / resolve_small_area_bytes(n);
    return (int)(k < least ? least : (k > most ? most : k));
}

size_t resolve_lanes_lds_bytes(int n, int Nx, int Ny) { return resolve_group_bytes(n, Nx, Ny) + sizeof(LdsR<double, 64>); }

static int cu_count() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        hipDeviceProp_t prop;
        cached[dev] = (hipGetDeviceProperties(&prop, dev) == hipSuccess && prop.multiProcessorCount > 0)
                          ? prop.multiProcessorCount : 256;
    }
    return cached[dev];
}
template <typename K> static int occupancy_blocks(K kernel, int threads, size_t lds) {
    int b = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, kernel, threads, lds) != hipSuccess || b < 1) b = 1;
    return b;
}
// One persistent launch over the jobs of pa (all of class cls).  sched: 0
// = default (one full residency of the kernel, grab 4), else
// (waves_per_cu << 8 | grab).
template <typename T, typename Tg>
static void launch_persistent(PersistArgs pa, int cls, int mode, int sched, hipStream_t s) {
    int grab = 4, waves_cu = 0;
    if (sched) {
        waves_cu = sched >> 8;
        grab = sched & 0xff;
    }
    pa.grab = grab;
    int units = 0;
    size_t lds = 0;
    for (int j = 0; j < pa.njobs; ++j) {
        const int u = pa.job[j].slots;
        units += u;
        pa.unit_end[j] = units;
        lds = std::max<size_t>(lds, pa.job[j].group_bytes);
    }
    if (units == 0) return;
    clear_counter(pa.queue, s);
    const int cus = cu_count();
    auto grid_for = [&](auto kernel, int threads, size_t dyn) {
        const int per_cu = waves_cu ? std::max(1, waves_cu / (threads / 64)) : occupancy_blocks(kernel, threads, dyn);
        return dim3((unsigned)std::min<long long>((long long)per_cu * cus, (units + grab - 1) / grab));
    };
    if (cls == 2) {   // complex64 coherence in the mixed precisions, complex128 in FP64
        if constexpr (sizeof(T) == sizeof(Tg)) {
            auto k = solve_generic_persistent<T, Tg, 1>;
            hipLaunchKernelGGL(k, grid_for(k, 128, lds), dim3(128), lds, s, pa);
        }
        return;
    }
    if (cls == 3) {   // complex128 coherence (FP64 Gram) in every precision
        if constexpr (sizeof(Tg) == 8) {
            auto k = solve_generic_persistent<T, Tg, 2>;
            hipLaunchKernelGGL(k, grid_for(k, 128, lds), dim3(128), lds, s, pa);
        }
        return;
    }
    if constexpr (sizeof(T) == sizeof(Tg)) {
        if (mode == 0) {
            auto k = solve_reg_persistent<T, Tg, MODE_EMI, 64>;
            hipLaunchKernelGGL(k, grid_for(k, 64, 0), dim3(64), 0, s, pa);
        } else if (mode == 2) {
            auto k = solve_reg_persistent<T, Tg, MODE_MLE, 64>;
            hipLaunchKernelGGL(k, grid_for(k, 64, 0), dim3(64), 0, s, pa);
        } else {
            auto k = solve_reg_persistent<T, Tg, MODE_EVD, 64>;
            hipLaunchKernelGGL(k, grid_for(k, 64, 0), dim3(64), 0, s, pa);
        }
    }
}

void launch_persistent_any(const PersistArgs& pa, int cls, int mode, int precision, int sched, hipStream_t s) {
    if (precision == FRINGE_PREC_FP64) launch_persistent<double, double>(pa, cls, mode, sched, s);
    else if (cls == 3) launch_persistent<float, double>(pa, cls, mode, sched, s);
    else launch_persistent<float, float>(pa, cls, mode, sched, s);
}
void resolve_tile(const LinkPlan& P, const float2* slc, const uint32_t* wts, float2* phase, float* tcorr,
                         float2* comp, hipStream_t s) {
    StageScope sc(STAGE_RESOLVE, s);
    SolveArgs a{};
    a.slc = slc;
    a.npx = P.npx;
    a.n = P.n;
    a.module = P.module;
    a.method = P.method;
    a.ref = P.ref;
    a.bw = P.bw;
    a.phase = phase;
    a.tcorr = tcorr;
    a.comp = comp;
    launch_resolve(P, wts, a, s);
}
}  // namespace fringe
