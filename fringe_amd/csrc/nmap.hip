// nmap.hip -- SHP (statistically homogeneous pixel) map on gfx950.
//
// Semantics follow src/nmap/nmap.cpp:204-233 and :345-473 with the
// race-free definition of the sweep (every pixel evaluates its own full
// window and writes only its own bits and count, as nmap_cuda.cu:259-334
// does): bits and counts are bit-exact against that definition.
//
// Stage 1 (nmap_prep): per pixel, amplitude |z| / alpha_b for every band,
// validity, and an ascending sort held in registers (bitonic network).
// Stage 2 (nmap_ks, nmap_walk): per pixel, the two-sample test against every
// valid in-image neighbour of the forward half of the window (dy > 0, or dy =
// 0 and dx >= 0), as the reference's sweep visits pairs (nmap.cpp:404-457); the
// bits go to a workspace.  Stage 3
// (nmap_mirror) assembles every output pixel's full mask: bit (dy, dx) of
// the backward half is bit (-dy, -dx) of neighbour p + (dy, dx), i.e. the
// same test of the same ordered pair, so each pair is tested once.  KS2: the
// statistic as an integer count k = D*n, compared with the largest one whose
// p-value reaches the threshold (found on the host).  AD2: the standardised
// Anderson-Darling statistic in double, bit-identical to the host's, compared
// with the largest statistic whose interpolated p-value still reaches the
// threshold (found on the host, so no exp/log runs on the device).
#include <algorithm>

#include "device_common.hpp"
#include "engine_internal.hpp"
#include "timing.hpp"

namespace fringe {

// |z| exactly as glibc's hypotf computes it for finite input (the value
// std::abs(std::complex<float>) returns on the host): the double-precision
// hypotenuse rounded once to float.  Non-finite parts give +inf when either
// part is infinite, NaN otherwise.
__device__ inline float amp_hypot(float x, float y) {
    if (!isfinite(x) || !isfinite(y)) {
        if (isinf(x) || isinf(y)) return INFINITY;
        return x + y;
    }
    double dx = (double)x, dy = (double)y;
    return (float)__builtin_sqrt(dx * dx + dy * dy);
}

template <int NP> __device__ inline void bitonic_sort(float (&a)[NP]) {
#pragma unroll
    for (int k = 2; k <= NP; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
            for (int t = 0; t < NP / 2; ++t) {
                const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), l = i | j;
                const bool up = ((i & k) == 0);
                const float x = a[i], y = a[l];
                const float lo = fminf(x, y), hi = fmaxf(x, y);
                a[i] = up ? lo : hi;
                a[l] = up ? hi : lo;
            }
        }
    }
}

// One thread per pixel of the whole tile.  amp_sorted is date-planar,
// [rank][pixel], so neighbouring threads read and write neighbouring words.
template <int NP>
__global__ __launch_bounds__(256) void nmap_prep(const NmapPlan P, const float2* __restrict__ slc,
                                                 const uint8_t* __restrict__ mask) {
    const long long npx = (long long)P.rows * P.cols;
    const int n = P.n;
    float* __restrict__ amp_sorted = P.d_amp;
    uint8_t* __restrict__ valid = P.d_valid;
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npx) return;
    float a[NP];
    bool ok = mask ? (mask[p] != 0) : true;
#pragma unroll
    for (int b = 0; b < NP; ++b) {
        a[b] = INFINITY;
        if (b < n) {
            const float2 z = slc[(long long)b * npx + p];
            const float val = (float)((double)amp_hypot(z.x, z.y) / P.alpha[b]);
            ok = ok && (val != 0.0f) && !isnan(val);
            a[b] = val;
        }
    }
    valid[p] = ok ? 1 : 0;
    if (!ok) return;
    bitonic_sort<NP>(a);
#pragma unroll
    for (int b = 0; b < NP; ++b)
        if (b < n) amp_sorted[(long long)b * npx + p] = a[b];
}

// term(j, m) = (2n m - n (j+1))^2 / ((j+1)(2n - j - 1)); every intermediate
// is an exact integer in double, so the one rounding is the division's.
__global__ void ad2_terms(double* __restrict__ T, int n) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (2 * n - 1) * (n + 1)) return;
    const int j = idx / (n + 1), m = idx % (n + 1);
    const double nsum = 2.0 * n, bj = j + 1;
    const double t = nsum * m - (double)n * bj;
    T[idx] = t * t / (bj * (nsum - bj));
}

__device__ inline double ad2_standardise(double S, int n, double sigma) {
    double A = 0.0;
    A = A + S / (n * 1.0);
    A = A + S / (n * 1.0);
    A = A / (2.0 * n);
    return (A - 1) / sigma;
}

// Forward-half words of the pixels of rows [fwd_row0, row_end): the output
// rows and the Ny rows above them whose forward tests reach into them.  Word w
// of pixel (r, c)'s mask (centre/32 .. nul-1) is in plane w - centre/32 of F, at
// (r - fwd_row0) * cols + c, as is its forward count (centre included) in fcnt.
__device__ inline int fwd_row0(const NmapPlan& P) { return max(0, P.row_begin - P.Ny); }
__device__ inline int centre_flat(const NmapPlan& P) { return P.Ny * (2 * P.Nx + 1) + P.Nx; }

// KS2: max |F_a - F_b| n <= K for ascending a and b if and only if
// b_{i-K} <= a_i and a_{i-K} <= b_i for every i in K .. n-1 (the count of a's
// values up to a_i is i + 1 at least, so that of b's has to be i + 1 - K).  So
// every date of a neighbour has a range, a_{i-K} <= b_i <= a_{i+K}, in which
// the pixel's own values, shifted by K, put it: one subtraction and one
// unsigned comparison a date, no merge.
//
// A workgroup takes up to 256 pixels of a row.  Per window row (and strip of
// 32 columns, and chunk of CH dates) the neighbours' samples are staged in
// LDS, pixel-major (a pitch of an odd number of quads: 16-byte reads without
// bank conflicts), and every thread tests its window columns from there; the ranges
// stay in registers.  Bound by the vector unit and the LDS reads (2.5 CH
// instructions and 4 CH bytes a pair).  2048 x 2048 pixels of 30 dates, 15 x 11
// window, against the register merge network it replaced: 16.1 -> 1.5 ms.
//
// Narrow images (NARROW, up to 32 columns) are taken as whole rows, as many as
// 256 threads hold: with a workgroup a row most lanes idle.  Maps of 30 dates,
// 15 x 11 window: 40000 x 1 pixels 2.39 -> 0.08 ms, 8000 x 8 0.56 -> 0.11, 5000 x
// 16 0.39 -> 0.13; from 33 columns on half of the lanes work either way.
template <int CH, bool NARROW>
__global__ __launch_bounds__(256) void nmap_ks(const NmapPlan P, int row_blocks, int wg0, uint32_t* __restrict__ F,
                                               int32_t* __restrict__ fcnt) {
    constexpr int PITCH = CH % 8 == 4 ? CH : CH + 4, STRIP = 32;
    __shared__ __align__(16) uint32_t L[(256 + STRIP - 1) * PITCH];
    const uint32_t* __restrict__ keys = reinterpret_cast<const uint32_t*>(P.d_amp);
    const uint8_t* __restrict__ valid = P.d_valid;
    const int n = P.n, rows = P.rows, cols = P.cols, Nx = P.Nx, Ny = P.Ny, nul = P.nul, K = P.ks_max;
    const long long npx = (long long)rows * cols;
    const int T = blockDim.x, tid = threadIdx.x;
    // blocks are dealt to the 8 XCDs round-robin: each takes a contiguous run
    // of rows, whose neighbours' samples stay in its L2
    const unsigned nb = gridDim.x, xcd = blockIdx.x % 8u;
    const int id = wg0 + (int)(xcd * (nb / 8u) + min(xcd, nb % 8u) + blockIdx.x / 8u);
    const int h0 = fwd_row0(P), at = NARROW ? tid / cols : 0;   // row in the workgroup
    const int r0 = h0 + (NARROW ? id * (T / cols) : id / row_blocks), r = r0 + at;
    const int c0 = NARROW ? 0 : id % row_blocks * T, c = NARROW ? tid - at * cols : c0 + tid;
    const bool here = NARROW ? at < T / cols && r < P.row_end : c < cols;
    const long long p = here ? (long long)r * cols + c : (long long)r0 * cols;
    const bool pv = here && valid[p] != 0;
    const int centre = centre_flat(P), fw = centre >> 5, nf = nul - fw;
    const long long plane = (long long)(P.row_end - h0) * cols;
    uint32_t* out = F + (p - (long long)h0 * cols);
    uint32_t lo[CH], span[CH];
    auto ranges = [&](int d0) {   // of dates d0 .. d0 + CH - 1; any valid key where there is none
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int d = d0 + i;
            lo[i] = d < n && d >= K ? keys[(long long)(d - K) * npx + p] : 0u;
            const uint32_t hi = d < n - K ? keys[(long long)(d + K) * npx + p] : 0x7FFFFFFFu;
            span[i] = hi - lo[i];
        }
    };
    const bool one = n <= CH;   // all dates in one chunk
    if (K >= 0 && one) ranges(0);
    int cnt = 0, word = 0, pos = centre & 31;
    uint64_t cur = 0;
    for (int dy = 0; dy <= Ny; ++dy) {
        for (int dx0 = dy == 0 ? 0 : -Nx; dx0 <= Nx; dx0 += STRIP) {
            const int w = min(STRIP, Nx - dx0 + 1);
            // positions that some column has (the others are outside the image)
            const int k0 = NARROW ? max(0, 1 - cols - dx0) : 0, k1 = NARROW ? min(w, cols - dx0) : w;
            uint32_t fail = NARROW ? ~0u : 0u;
            if (r0 + dy < rows && K >= 0) {   // uniform
                for (int d0 = 0; d0 < n; d0 += CH) {
                    const int m = min(CH, n - d0);
                    __syncthreads();   // the last strip's reads are over
                    for (int e = tid; e < (NARROW ? T / cols * cols : T + w - 1); e += T) {
                        const int er = NARROW ? e / cols : 0, cc = NARROW ? e - er * cols : c0 + dx0 + e, rr = r0 + er + dy;
                        const bool in = cc >= 0 && cc < cols && (!NARROW || rr < rows);
                        const long long q = in ? (long long)rr * cols + cc : 0;
                        const bool ok = in && valid[q] != 0;
#pragma unroll
                        for (int i = 0; i < CH; i += 4) {
                            uint32_t v[4];
#pragma unroll
                            for (int u = 0; u < 4; ++u) v[u] = i + u < m ? keys[(long long)(d0 + i + u) * npx + q] : 0u;
                            // no range holds the key of a pixel that is not there
                            *(uint4*)&L[e * PITCH + i] = ok ? make_uint4(v[0], v[1], v[2], v[3])
                                                            : make_uint4(~0u, ~0u, ~0u, ~0u);
                        }
                    }
                    __syncthreads();
                    if (!one) ranges(d0);
#pragma unroll 2
                    for (int k = k0; k < k1; ++k) {
                        const bool in = !NARROW || (c + dx0 + k >= 0 && c + dx0 + k < cols);
                        const int e = NARROW ? (in ? tid + dx0 + k : 0) : tid + k;
                        uint32_t over = in ? 0u : 1u;   // what exceeds a range (saturating)
#pragma unroll
                        for (int i = 0; i < CH; i += 4) {
                            const uint4 b = *(const uint4*)&L[e * PITCH + i];
                            over |= __builtin_elementwise_sub_sat(b.x - lo[i], span[i]);
                            over |= __builtin_elementwise_sub_sat(b.y - lo[i + 1], span[i + 1]);
                            over |= __builtin_elementwise_sub_sat(b.z - lo[i + 2], span[i + 2]);
                            over |= __builtin_elementwise_sub_sat(b.w - lo[i + 3], span[i + 3]);
                        }
                        if (NARROW && d0 == 0) fail &= ~(1u << k);
                        fail |= (over != 0u ? 1u : 0u) << k;
                    }
                }
            } else {
                fail = ~0u;
            }
            uint32_t bits = pv ? ~fail & (~0u >> (32 - w)) : 0u;
            if (dy == 0 && dx0 == 0) bits |= pv ? 1u : 0u;   // the pixel itself
            cnt += __popc(bits);
            cur |= (uint64_t)bits << pos;
            pos += w;
            if (pos >= 32) {
                if (here) out[word * plane] = (uint32_t)cur;
                ++word;
                cur >>= 32;
                pos -= 32;
            }
        }
    }
    if (here) {
        for (; word < nf; ++word) {
            out[word * plane] = (uint32_t)cur;
            cur = 0;
        }
        fcnt[p - (long long)h0 * cols] = cnt;
    }
}

// AD2: the merge as a walk.  The inner sum of AD2unique::test
// (AD2unique.hpp:206-351) merges ascending a (the pixel, the test's first
// sample) and b with ties taken from b first and adds, for every merged
// position j < 2n-1, the term of (j, m_j) where m_j counts the a values among
// the first j+1; the same values are added here in the same order.  The term
// depends on |2 m - (j+1)| alone, so half of the table is kept.
//
// A workgroup takes 64 pixels of a row; per window row (and strip of 32
// columns) the neighbours' samples are staged in LDS next to the pixels' own
// and the terms, and its four waves share the window's columns, two walks at
// a time per thread.  Bound by the walk's chain (compare, address, LDS read).
// 203 x 317 pixels of 72 dates, 13 x 9 window, against one thread per pixel
// walking in global memory (one wave per SIMD): 3.6 -> 0.6 ms; 512 x 512
// pixels of 30 dates against a merge network in registers: 1.90 -> 0.72.
constexpr int kWalkStrip = 32;
__host__ __device__ inline int ad2_row_terms(int n, int b) { return (b < 2 * n - b ? b : 2 * n - b) / 2 + 1; }   // of position b - 1
__host__ __device__ inline int ad2_row_offset(int n, int b) {   // sum of ad2_row_terms(n, 1 .. b - 1)
    const int t = b <= n ? b - 1 : n, u = 2 * n - b;
    const int head = t * t / 4 + t;
    return b <= n ? head : head + (n - 1) * (n - 1) / 4 - u * u / 4 + (b - 1 - n);
}
static size_t ad2_walk_bytes(int n) {
    return (size_t)ad2_row_offset(n, 2 * n) * 8 + (size_t)((64 + 64 + kWalkStrip - 1) * ((n + 1) | 1) + 4 * 64) * 4;
}

// Narrow images as in nmap_ks: maps of 30 dates, 40000 x 1 pixels 6.87 -> 0.12
// ms, 8000 x 8 1.56 -> 0.30, 5000 x 16 1.02 -> 0.35.
template <bool NARROW>
__global__ __launch_bounds__(256) void nmap_walk(const NmapPlan P, int row_blocks, int wg0, uint32_t* __restrict__ F,
                                                 int32_t* __restrict__ fcnt) {
    extern __shared__ __align__(16) char smem[];
    const uint32_t* __restrict__ keys = reinterpret_cast<const uint32_t*>(P.d_amp);
    const uint8_t* __restrict__ valid = P.d_valid;
    const int n = P.n, rows = P.rows, cols = P.cols, Nx = P.Nx, Ny = P.Ny, nul = P.nul;
    const int pitch = (n + 1) | 1;   // a run's keys, then one above every amplitude
    const int terms = ad2_row_offset(n, 2 * n);
    double* T = (double*)smem;
    uint32_t* own = (uint32_t*)(T + terms);
    uint32_t* oth = own + 64 * pitch;
    uint32_t* part = oth + (64 + kWalkStrip - 1) * pitch;   // [4][64] bits of the waves
    const long long npx = (long long)rows * cols;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned nb = gridDim.x, xcd = blockIdx.x % 8u;   // as nmap_ks
    const int id = wg0 + (int)(xcd * (nb / 8u) + min(xcd, nb % 8u) + blockIdx.x / 8u);
    const int h0 = fwd_row0(P), at = NARROW ? lane / cols : 0;   // row in the workgroup
    const int r0 = h0 + (NARROW ? id * (64 / cols) : id / row_blocks), r = r0 + at;
    const int c0 = NARROW ? 0 : id % row_blocks * 64, c = NARROW ? lane - at * cols : c0 + lane;
    const bool here = NARROW ? at < 64 / cols && r < P.row_end : c < cols;
    const long long p = here ? (long long)r * cols + c : (long long)r0 * cols;
    const bool pv = here && valid[p] != 0;
    const int centre = centre_flat(P), fw = centre >> 5, nf = nul - fw;
    const long long plane = (long long)(P.row_end - h0) * cols;
    uint32_t* out = F + (p - (long long)h0 * cols);
    for (int j = wave; j < 2 * n - 1; j += 4) {
        const int b = j + 1, at = ad2_row_offset(n, b);
        for (int d = lane; d < ad2_row_terms(n, b); d += 64) T[at + d] = P.d_ad2[j * (n + 1) + (b + 2 * d + (b & 1)) / 2];
    }
    // keys of 64 or more consecutive pixels of row `row` from column `from` on,
    // or of the rows from it on
    auto stage = [&](uint32_t* dst, int row, int from, int count) {
        for (int e = lane; e < count; e += 64) {
            const int er = NARROW ? e / cols : 0, rr = row + er, cc = NARROW ? e - er * cols : from + e;
            const bool in = cc >= 0 && cc < cols && (!NARROW || (er < 64 / cols && rr < rows));
            const long long q = in ? (long long)rr * cols + cc : 0;
            const bool ok = in && valid[q] != 0;
            for (int i = wave; i <= n; i += 4) dst[e * pitch + i] = ok && i < n ? keys[(long long)i * npx + q] : ~0u;
        }
    };
    stage(own, r0, c0, 64);
    int cnt = 0, word = 0, pos = centre & 31;
    uint64_t cur = 0;
    for (int dy = 0; dy <= Ny; ++dy) {
        for (int dx0 = dy == 0 ? 0 : -Nx; dx0 <= Nx; dx0 += kWalkStrip) {
            const int w = min(kWalkStrip, Nx - dx0 + 1);
            if (r0 + dy < rows) stage(oth, r0 + dy, c0 + dx0, NARROW ? 64 : 64 + w - 1);
            __syncthreads();
            uint32_t bits = 0u;
            if (r0 + dy < rows)
                // (positions that some column has)
                for (int k0 = wave + (NARROW ? max(0, 1 - cols - dx0) : 0); k0 < (NARROW ? min(w, cols - dx0) : w); k0 += 8) {
                    const uint32_t *pa[2], *pb[2];
                    uint32_t x[2], y[2];
                    int dd[2] = {0, 0};
                    double S[2] = {0.0, 0.0};
                    bool there[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int k = k0 + 4 * u < w ? k0 + 4 * u : k0;   // (once more where there is no second)
                        const bool in = !NARROW || (c + dx0 + k >= 0 && c + dx0 + k < cols);
                        pa[u] = own + lane * pitch;
                        pb[u] = oth + (NARROW ? (in ? lane + dx0 + k : lane) : lane + k) * pitch;
                        x[u] = *pa[u];
                        y[u] = *pb[u];
                        there[u] = in && y[u] != ~0u && x[u] != ~0u;
                        // for a neighbour that is not there, the pixel's run twice (if
                        // that is not there either, words of other runs: not used)
                        if (!there[u]) pb[u] = pa[u], y[u] = x[u];
                    }
                    const double* row = T;
                    for (int b = 1; b < 2 * n; ++b) {
                        const int odd = b & 1;
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const bool take_a = x[u] < y[u];
                            pa[u] += take_a ? 1 : 0;
                            pb[u] += take_a ? 0 : 1;
                            const uint32_t v = *(take_a ? pa[u] : pb[u]);
                            x[u] = take_a ? v : x[u];
                            y[u] = take_a ? y[u] : v;
                            dd[u] += take_a ? 1 : -1;
                            S[u] = S[u] + row[(abs(dd[u]) - odd) >> 1];
                        }
                        row += ad2_row_terms(n, b);
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        if (there[u] && k0 + 4 * u < w && ad2_standardise(S[u], n, P.ad2_sigma) <= P.ad2_max)
                            bits |= 1u << (k0 + 4 * u);
                }
            part[tid] = bits;
            __syncthreads();   // the strip's reads are over, too
            bits = pv ? part[lane] | part[64 + lane] | part[128 + lane] | part[192 + lane] : 0u;
            if (dy == 0 && dx0 == 0) bits |= pv ? 1u : 0u;   // the pixel itself
            cnt += __popc(bits);
            cur |= (uint64_t)bits << pos;
            pos += w;
            if (pos >= 32) {
                if (here && wave == 0) out[word * plane] = (uint32_t)cur;
                ++word;
                cur >>= 32;
                pos -= 32;
            }
        }
    }
    if (here && wave == 0) {
        for (; word < nf; ++word) {
            out[word * plane] = (uint32_t)cur;
            cur = 0;
        }
        fcnt[p - (long long)h0 * cols] = cnt;
    }
}

// Full masks of the output rows.  Backward position flat (< centre) of
// pixel p holds the forward bit W-1-flat of q = p + (dy, dx), the pair's
// one test; q lies in rows [fwd_row0, row_end) whenever it is in the image.
__global__ __launch_bounds__(256) void nmap_mirror(const NmapPlan P, const uint32_t* __restrict__ F,
                                                   const int32_t* __restrict__ fcnt, uint32_t* __restrict__ wts,
                                                   int32_t* __restrict__ count) {
    const int cols = P.cols, Nx = P.Nx, Ny = P.Ny, nul = P.nul;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)(P.row_end - P.row_begin) * cols) return;
    const int r = P.row_begin + (int)(t / cols);
    const int c = (int)(t % cols);
    const int h0 = fwd_row0(P);
    const int centre = centre_flat(P), fw = centre >> 5, nf = nul - fw;
    const int last = (2 * Ny + 1) * (2 * Nx + 1) - 1;
    const long long plane = (long long)(P.row_end - h0) * cols, fp = (long long)(r - h0) * cols + c;
    uint32_t* out = wts + ((long long)r * cols + c) * nul;
    int cnt = fcnt[fp];
    int word = 0, flat = 0;
    uint32_t cur = 0u;
    for (int dy = -Ny; dy <= 0; ++dy) {
        const int rr = r + dy;
        for (int dx = -Nx; dx <= (dy == 0 ? -1 : Nx); ++dx, ++flat) {
            if ((flat >> 5) != word) {
                out[word] = cur;
                cur = 0u;
                word = flat >> 5;
            }
            const int cc = c + dx;
            if (rr < 0 || cc < 0 || cc >= cols) continue;
            const int mf = last - flat;
            const uint32_t qw = F[((mf >> 5) - fw) * plane + (long long)(rr - h0) * cols + cc];
            if ((qw >> (mf & 31)) & 1u) {
                cur |= (1u << (flat & 31));
                ++cnt;
            }
        }
    }
    // flat == centre: the rest comes from the pixel's own forward words
    if (fw != word) {
        out[word] = cur;
        cur = 0u;
    }
    const uint32_t* mine = F + fp;
    out[fw] = cur | mine[0];
    for (int i = 1; i < nf; ++i) out[fw + i] = mine[i * plane];
    count[(long long)r * cols + c] = cnt;
}

int nmap_fwd_words(int Nx, int Ny) { return shp_words(Nx, Ny) - ((Ny * (2 * Nx + 1) + Nx) >> 5); }

template <int NP>
static void launch_prep(const NmapPlan& P, const float2* slc, const uint8_t* mask, hipStream_t s) {
    const long long npx = (long long)P.rows * P.cols;
    const int threads = 256;
    const long long blocks = (npx + threads - 1) / threads;
    hipLaunchKernelGGL(nmap_prep<NP>, dim3((unsigned)blocks), dim3(threads), 0, s, P, slc, mask);
}

// Images up to kNarrow columns are mapped row after row.
constexpr int kNarrow = 32;
// A launch holds less than 2^32 threads: launch(first, count) for parts of
// `wgs` workgroups.
template <typename L> static void in_parts(long long wgs, int threads, L launch) {
    const long long most = ((1ll << 32) - 1) / threads;
    for (long long w = 0; w < wgs; w += most) launch((int)w, dim3((unsigned)std::min(wgs - w, most)));
}

template <int CH> static void launch_ks(const NmapPlan& P, long long fwd_rows, hipStream_t s) {
    if (P.cols <= kNarrow) {
        const int per = 256 / P.cols;
        in_parts((fwd_rows + per - 1) / per, 256, [&](int wg0, dim3 grid) {
            hipLaunchKernelGGL((nmap_ks<CH, true>), grid, dim3(256), 0, s, P, 1, wg0, P.d_fwd, P.d_fcnt);
        });
        return;
    }
    // the fewest workgroups of at most four waves, of the fewest waves
    const int waves = (P.cols + 63) / 64, blocks = (waves + 3) / 4, per = (waves + blocks - 1) / blocks;
    in_parts(fwd_rows * blocks, 64 * per, [&](int wg0, dim3 grid) {
        hipLaunchKernelGGL((nmap_ks<CH, false>), grid, dim3(64 * per), 0, s, P, blocks, wg0, P.d_fwd, P.d_fcnt);
    });
}

static void launch_walk(const NmapPlan& P, long long fwd_rows, hipStream_t s) {
    const size_t lds = ad2_walk_bytes(P.n);
    if (P.cols <= kNarrow) {
        const int per = 64 / P.cols;
        in_parts((fwd_rows + per - 1) / per, 256, [&](int wg0, dim3 grid) {
            hipLaunchKernelGGL(nmap_walk<true>, grid, dim3(256), lds, s, P, 1, wg0, P.d_fwd, P.d_fcnt);
        });
        return;
    }
    const int blocks = (P.cols + 63) / 64;
    in_parts(fwd_rows * blocks, 256, [&](int wg0, dim3 grid) {
        hipLaunchKernelGGL(nmap_walk<false>, grid, dim3(256), lds, s, P, blocks, wg0, P.d_fwd, P.d_fcnt);
    });
}

int nmap_launch(const NmapPlan& P, const float2* slc, const uint8_t* mask, uint32_t* wts,
                int32_t* count, hipStream_t s) {
    {
        StageScope sc(STAGE_NMAP_PREP, s);
        if (P.n <= 8) launch_prep<8>(P, slc, mask, s);
        else if (P.n <= 16) launch_prep<16>(P, slc, mask, s);
        else if (P.n <= 32) launch_prep<32>(P, slc, mask, s);
        else if (P.n <= 64) launch_prep<64>(P, slc, mask, s);
        else launch_prep<128>(P, slc, mask, s);
    }
    const long long nout = (long long)(P.row_end - P.row_begin) * P.cols;
    if (nout > 0) {
        const int threads = 256;
        // forward halves of the output rows and of the Ny rows above them
        const int h0 = P.row_begin - P.Ny > 0 ? P.row_begin - P.Ny : 0;
        StageScope sc(STAGE_NMAP_KS, s);
        if (P.method == 0) {
            // chunks of at most 32 dates, alike and padded to quads
            const int chunks = (P.n + 31) / 32, quads = ((P.n + chunks - 1) / chunks + 3) / 4;
            const int fr = P.row_end - h0;
            switch (quads) {
                case 1: launch_ks<4>(P, fr, s); break;
                case 2: launch_ks<8>(P, fr, s); break;
                case 3: launch_ks<12>(P, fr, s); break;
                case 4: launch_ks<16>(P, fr, s); break;
                case 5: launch_ks<20>(P, fr, s); break;
                case 6: launch_ks<24>(P, fr, s); break;
                case 7: launch_ks<28>(P, fr, s); break;
                default: launch_ks<32>(P, fr, s); break;
            }
        } else {
            const int nt = (2 * P.n - 1) * (P.n + 1);
            hipLaunchKernelGGL(ad2_terms, dim3((nt + 255) / 256), dim3(256), 0, s, P.d_ad2, P.n);
            launch_walk(P, P.row_end - h0, s);
        }
        hipLaunchKernelGGL(nmap_mirror, dim3((unsigned)((nout + threads - 1) / threads)), dim3(threads), 0, s,
                           P, (const uint32_t*)P.d_fwd, (const int32_t*)P.d_fcnt, wts, count);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fringe
