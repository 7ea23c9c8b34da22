// link.hip -- per-pixel phase linking on gfx950: the FP64 ("plain") masked-
// neighbourhood coherence, and the rounds of Gram and solver launches of a
// tile and of a batch of tiles.
//
// Reference semantics: src/evd/evd.cpp:512-788 (EVD / MLE / STBAS) and
// src/phase_link/phase_link.cpp:479-666 (EMI with EVD fallback).  The LAPACK
// calls of EigenLapack.hpp (zheevr RANGE='I', zpotrf + zpotri) are replaced by
// the solvers of solvers.hip.
#include <algorithm>

#include "device_common.hpp"
#include "engine_internal.hpp"
#include "link_solve.hpp"
#include "timing.hpp"

namespace fringe {

// ---------------------------------------------------------------------------
// FP64 Gram over a chunk of output pixels, one group of G lanes per pixel
// (the per-pixel body is gram_f64_pixel in gram64.hpp).
// ---------------------------------------------------------------------------
template <int G, int R, int CB>
__global__ __launch_bounds__(64) void gram_f64(GramArgs a) {
    constexpr int GPW = 64 / G;
    const int grp = threadIdx.x / G, g = threadIdx.x % G;
    const int slot = blockIdx.x * GPW + grp;
    extern __shared__ __align__(16) char smem[];
    const bool inslot = slot < a.slots;
    const long long pix = a.first + (inslot ? slot : 0);
    cx<double>* gam = (cx<double>*)a.gamma + (size_t)(inslot ? slot : 0) * a.n * a.n;
    const int np = gram_f64_pixel<G, R, CB>(a, inslot, pix, gam, smem + grp * a.group_bytes);
    if (inslot && g == 0) a.npix[slot] = np;
}

template <int G, int R, int CB>
static void launch_gram_f64(GramArgs a, hipStream_t s) {
    constexpr int GPW = 64 / G;
    a.group_bytes = gram_f64_group_bytes(a.n, a.Nx, a.Ny, CB);
    const unsigned blocks = (unsigned)((a.slots + GPW - 1) / GPW);
    hipLaunchKernelGGL((gram_f64<G, R, CB>), dim3(blocks), dim3(64), a.group_bytes * GPW, s, a);
}

// The FP64 coherence of a.slots slots: on the matrix cores where the FP64
// solver is (n <= 128 by default; the re-solve uses the same Gram as the plain
// path either way), else one group of lanes per pixel.
static void gram_f64_slots(const GramArgs& g, hipStream_t s) {
    if (matrix_solver_selected(g.n, FRINGE_PREC_FP64)) launch_gram_mfma64(g, s);
    else if (g.n <= 64) launch_gram_f64<64, 1, 32>(g, s);
    else if (g.n <= 128) launch_gram_f64<64, 2, 16>(g, s);
    else launch_gram_f64<64, 4, 16>(g, s);
}

__global__ void zero_i32(int* p, int count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = 0;
}
void clear_counter(int* p, hipStream_t s) { hipLaunchKernelGGL(zero_i32, dim3(1), dim3(64), 0, s, p, 1); }

bool link_uses_mfma(int n, int precision) { return precision != FRINGE_PREC_FP64 && n <= kMaxBandsMfma; }
bool link_certifies(int n, int precision) { return precision != FRINGE_PREC_FP64; }

size_t link_gamma_bytes_per_pixel(int n, int precision) {
    const size_t e = link_uses_mfma(n, precision) ? 8 : 16;
    return (size_t)n * n * e + sizeof(int);
}

// Coherence matrices only (the Gram stage of link_launch), into a caller
// buffer covering the output rows: complex64 from the MFMA Gram, complex128
// from the FP64 one.
int coherence_launch(const LinkPlan& P, const float2* slc, const uint32_t* wts, void* gamma, int* npix,
                     hipStream_t s) {
    const long long first = (long long)P.row_begin * P.cols;
    const int slots = (P.row_end - P.row_begin) * P.cols;
    if (slots <= 0) return 0;
    if (link_uses_mfma(P.n, P.precision)) {
        if (pack_launch(slc, P.rows, P.cols, P.n, P.precision != FRINGE_PREC_MIXED_BF16, P.d_pack, nullptr, s) != 0)
            return -1;
        LinkPlan Q = P;
        Q.d_gamma = gamma;
        Q.d_npix = npix;
        return gram_mfma_launch(Q, P.d_pack, wts, first, slots, s);
    }
    GramArgs g{};
    g.slc = slc;
    g.wts = wts;
    g.rows = P.rows;
    g.cols = P.cols;
    g.n = P.n;
    g.Nx = P.Nx;
    g.Ny = P.Ny;
    g.nul = P.nul;
    g.min_nb = P.min_nb;
    g.npx = P.npx;
    g.first = first;
    g.slots = slots;
    g.gamma = gamma;
    g.npix = npix;
    gram_f64_slots(g, s);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------------------
// Pieces of a link: the Gram of a segment of whole rows, the solver launch
// (a grid, or a persistent queue of jobs), the FP64 re-solve of a tile.
// ---------------------------------------------------------------------------
static void gram_segment(const LinkPlan& P, const float2* slc, const uint32_t* wts, long long first, int slots,
                         void* gamma, int* npix, hipStream_t s, int* rc) {
    if (!link_uses_mfma(P.n, P.precision)) {
        GramArgs g{};
        g.slc = slc;
        g.wts = wts;
        g.rows = P.rows;
        g.cols = P.cols;
        g.n = P.n;
        g.Nx = P.Nx;
        g.Ny = P.Ny;
        g.nul = P.nul;
        g.min_nb = P.min_nb;
        g.npx = P.npx;
        g.first = first;
        g.slots = slots;
        g.gamma = gamma;
        g.npix = npix;
        gram_f64_slots(g, s);
    } else {
        LinkPlan Q = P;
        Q.d_gamma = gamma;
        Q.d_npix = npix;
        if (gram_mfma_launch(Q, P.d_pack, wts, first, slots, s) != 0) *rc = -1;
    }
}

// Date class of the vector-unit solvers (the matrix-core ones serve n <= 32
// and, by default, n <= 128): 1 one row per lane (n <= 64), 2 work matrix, one
// row per thread (n <= 128: the MFMA Gram's complex64 coherence in the mixed
// precisions), 3 two rows per thread (n > 128, complex128 coherence).
static int solve_class(int n) { return n <= 64 ? 1 : (n <= kMaxBandsMfma ? 2 : 3); }

static PJob make_job(const LinkPlan& P, const float2* slc, float2* phase, float* tcorr, float2* comp,
                     long long first, int slots, const void* gamma, const int* npix, void* awork, size_t awork_stride) {
    PJob J{};
    J.gamma = gamma;
    J.npix = npix;
    J.slc = slc;
    J.phase = phase;
    J.tcorr = tcorr;
    J.comp = comp;
    J.cert_list = P.d_cert_list;
    J.cert_count = P.d_cert_count;
    J.cert_cap = P.cert_cap;
    J.awork = awork;
    J.awork_stride = awork_stride;
    J.npx = P.npx;
    J.first = first;
    J.slots = slots;
    J.n = P.n;
    J.ref = P.ref;
    J.bw = P.bw;
    const bool f64 = P.precision == FRINGE_PREC_FP64;
    J.group_bytes = (unsigned)(f64 ? solve_group_bytes<double>(P.n, awork == nullptr)
                                   : solve_group_bytes<float>(P.n, awork == nullptr));
    return J;
}

int link_launch(const LinkPlan& P, const float2* slc, const uint32_t* wts, float2* phase,
                float* tcorr, float2* comp, hipStream_t s) {
    const long long first_out = (long long)P.row_begin * P.cols;
    const long long total = (long long)(P.row_end - P.row_begin) * P.cols;
    const bool fp64 = (P.precision == FRINGE_PREC_FP64);
    const bool mfma = link_uses_mfma(P.n, P.precision);
    const int mode = solve_mode_index(P.module, P.method);
    const int sched = schedule_lookup(FRINGE_SCHED_SOLVE, P.n, mode, fp64 ? 0 : 1, 0);
    if (mfma) {
        StageScope sc(STAGE_PACK, s);
        if (pack_launch(slc, P.rows, P.cols, P.n, P.precision != FRINGE_PREC_MIXED_BF16, P.d_pack, P.d_cert_count, s) != 0)
            return -1;
    } else if (P.d_cert_count) {
        clear_counter(P.d_cert_count, s);
    }
    int rc = 0;
    for (long long done = 0; done < total; done += P.chunk) {
        const int slots = (int)((total - done) < P.chunk ? (total - done) : P.chunk);
        const long long first = first_out + done;
        {
            StageScope sc(STAGE_GRAM, s);
            gram_segment(P, slc, wts, first, slots, P.d_gamma, P.d_npix, s, &rc);
            if (rc) return -1;
        }
        StageScope sc(STAGE_SOLVE, s);
        if (sched && P.d_queue && !matrix_solver_selected(P.n, P.precision)) {
            PersistArgs pa{};
            pa.module = P.module;
            pa.method = P.method;
            pa.njobs = 1;
            pa.queue = P.d_queue;
            pa.job[0] = make_job(P, slc, phase, tcorr, comp, first, slots, P.d_gamma, P.d_npix, P.d_awork,
                                 P.awork_stride);
            launch_persistent_any(pa, solve_class(P.n), mode, P.precision, sched, s);
        } else {
            SolveArgs a{};
            a.cert_list = P.d_cert_list;
            a.cert_count = P.d_cert_count;
            a.cert_cap = P.cert_cap;
            a.gamma = P.d_gamma;
            a.npix = P.d_npix;
            a.slc = slc;
            a.npx = P.npx;
            a.first = first;
            a.slots = slots;
            a.n = P.n;
            a.module = P.module;
            a.method = P.method;
            a.ref = P.ref;
            a.bw = P.bw;
            a.phase = phase;
            a.tcorr = tcorr;
            a.comp = comp;
            a.awork = P.d_awork;
            a.awork_stride = P.awork_stride;
            launch_solve(a, P.precision, s);
        }
        if (hipGetLastError() != hipSuccess) return -1;
    }
    if (P.d_cert_count) {
        resolve_tile(P, slc, wts, phase, tcorr, comp, s);
        if (hipGetLastError() != hipSuccess) return -1;
    }
    return 0;
}

// ---------------------------------------------------------------------------
// Batch of independent tiles (fringe_link_batch_run): rounds of coherence
// segments from several tiles in one buffer, one persistent solve launch
// per date class and round.
// ---------------------------------------------------------------------------
static SolveArgs solve_args_of(const PJob& J, int module, int method) {
    SolveArgs a{};
    a.gamma = J.gamma;
    a.npix = J.npix;
    a.slc = J.slc;
    a.npx = J.npx;
    a.first = J.first;
    a.slots = J.slots;
    a.n = J.n;
    a.module = module;
    a.method = method;
    a.ref = J.ref;
    a.bw = J.bw;
    a.phase = J.phase;
    a.tcorr = J.tcorr;
    a.comp = J.comp;
    a.cert_list = J.cert_list;
    a.cert_count = J.cert_count;
    a.cert_cap = J.cert_cap;
    a.awork = J.awork;
    a.awork_stride = J.awork_stride;
    return a;
}

int link_batch_launch(const BatchPlan& B, hipStream_t s) {
    const int count = (int)B.tiles.size();
    for (int i = 0; i < count; ++i) {
        const BatchTile& T = B.tiles[i];
        if (link_uses_mfma(T.P.n, T.P.precision)) {
            StageScope sc(STAGE_PACK, s);
            if (pack_launch(T.slc, T.P.rows, T.P.cols, T.P.n, T.P.precision != FRINGE_PREC_MIXED_BF16, T.P.d_pack,
                            T.P.d_cert_count, s) != 0)
                return -1;
        } else if (T.P.d_cert_count) {
            clear_counter(T.P.d_cert_count, s);
        }
    }
    const int mode = solve_mode_index(B.module, B.method);
    int item = 0;
    long long row = count ? B.tiles[0].P.row_begin : 0;
    int rc = 0;
    while (item < count) {
        // 0: the matrix-core solver's tiles, one grid launch each; 1..3: one
        // persistent launch per date class (solve_class)
        PersistArgs pa[4] = {};
        size_t off = 0;      // bytes of the round buffer in use
        long long soff = 0;  // slots in use
        bool full = false;
        while (item < count && !full) {
            const BatchTile& T = B.tiles[item];
            const LinkPlan& P = T.P;
            const int cls = matrix_solver_selected(P.n, P.precision) ? 0 : solve_class(P.n);
            const long long rem = P.row_end - row;
            if (rem <= 0) {
                ++item;
                if (item < count) row = B.tiles[item].P.row_begin;
                continue;
            }
            if (pa[cls].njobs == kMaxJobs) break;
            // bytes per row: coherence matrices, plus the work matrices above 64
            // dates when they live in global memory, each block 256-aligned
            const size_t per_row = (size_t)P.cols * (link_gamma_bytes_per_pixel(P.n, P.precision) - sizeof(int) +
                                                     P.awork_stride);
            long long rows = (long long)((B.round_bytes > off + 512 ? B.round_bytes - off - 512 : 0) / per_row);
            rows = std::min(rows, rem);
            const int th = link_uses_mfma(P.n, P.precision) ? gram_stage_rows(P.n, P.Nx, P.Ny) : 1;
            if (rows < rem && rows > th) rows -= rows % th;
            if (rows <= 0) {
                full = true;
                break;
            }
            const int slots = (int)(rows * P.cols);
            const long long first = row * P.cols;
            char* gam = (char*)B.d_round + off;
            const size_t gbytes = align256((size_t)slots * P.n * P.n * (link_uses_mfma(P.n, P.precision) ? 8 : 16));
            void* aw = nullptr;
            if (P.awork_stride) aw = gam + gbytes;
            int* npix = B.d_npix + soff;
            {
                StageScope sc(STAGE_GRAM, s);
                gram_segment(P, T.slc, T.wts, first, slots, gam, npix, s, &rc);
                if (rc) return -1;
            }
            pa[cls].job[pa[cls].njobs++] = make_job(P, T.slc, T.phase, T.tcorr, T.comp, first, slots, gam, npix, aw,
                                                    P.awork_stride);
            off += gbytes + (size_t)slots * P.awork_stride;
            soff += slots;
            row += rows;
        }
        StageScope sc(STAGE_SOLVE, s);
        for (int j = 0; j < pa[0].njobs; ++j)
            launch_solve(solve_args_of(pa[0].job[j], B.module, B.method), B.precision, s);
        for (int c = 1; c < 4; ++c) {
            if (!pa[c].njobs) continue;
            pa[c].module = B.module;
            pa[c].method = B.method;
            pa[c].queue = B.d_queue + c;
            const int sched = schedule_lookup(FRINGE_SCHED_SOLVE, c == 1 ? 64 : 256, mode,
                                              B.precision == FRINGE_PREC_FP64 ? 0 : 1, 0);
            if (pa[c].njobs == 1 && sched == 0) {
                // a lone job of its class: the launch the schedule prefers for one tile
                launch_solve(solve_args_of(pa[c].job[0], B.module, B.method), B.precision, s);
            } else {
                launch_persistent_any(pa[c], c, mode, B.precision, sched, s);
            }
        }
        if (hipGetLastError() != hipSuccess) return -1;
    }
    for (int i = 0; i < count; ++i) {
        const BatchTile& T = B.tiles[i];
        if (T.P.d_cert_count && T.P.row_end > T.P.row_begin) {
            LinkPlan Q = T.P;
            Q.d_rwork = B.d_rwork;
            resolve_tile(Q, T.slc, T.wts, T.phase, T.tcorr, T.comp, s);
            if (hipGetLastError() != hipSuccess) return -1;
        }
    }
    return 0;
}

}  // namespace fringe
