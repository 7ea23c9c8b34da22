// gram_mfma64.hpp -- FP64 masked-neighbourhood coherence of one pixel on the
// matrix cores, up to 128 dates (evd.cpp:530-582 / phase_link.cpp:496-538):
// the plain FP64 path's Gram, and the re-solve's.
//
// A workgroup of NW = ceil(n / 16) waves per pixel.  The masked, in-image
// window positions are compacted into a list; 16 of them at a time are staged
// in LDS (each wave its 16 dates), and per four positions wave w multiplies
// its dates with those of tile columns w, w + 1, ..., w + NW / 2 (modulo NW):
// four v_mfma_f64_16x16x4 a tile, k the positions.  Each pair of tiles is so
// computed once; the other one is its conjugate transpose.  Samples are
// widened to double, products and sums are FP64.
//
// Bound by the FP64 matrix instructions (whose rate is the vector unit's,
// but which need no operand from LDS per product).  Against the vector-unit
// Gram it replaced, 301 x 409 pixels of 27 dates (15 x 11 window, 80 % fill):
// 4.3 -> 1.7 ms.
#pragma once
#include "gram64.hpp"
#include "solve_mfma.hpp"

namespace fringe {

template <int NW> struct LdsGram64 {
    static constexpr int N = 16 * NW, S = N + 16;   // rows 32 banks apart
    float2 z[2][16][S];   // staged samples, [position][date]
    double dg[N];
    int cnt;
};

// Bytes of the position list (dynamic LDS).
inline __host__ __device__ size_t gram_list_bytes(int Nx, int Ny) {
    return (((size_t)(2 * Ny + 1) * (2 * Nx + 1) + 16) * 4 + 15) & ~(size_t)15;
}

// Coherence of pixel `pix` into gam[n][n] (both triangles, unit diagonal);
// returns the neighbour count, or -1 when the pixel is not linked (gam is
// then not written).  Every wave of the workgroup calls it; the caller
// synchronises before gam is read.
template <int NW>
__device__ __forceinline__ int gram_mfma64_pixel(const GramArgs& a, LdsGram64<NW>& L, int* list, int w, int lane,
                                                 long long pix, cx<double>* gam) {
    constexpr int T = NW / 2 + 1;   // tiles of a wave
    const int n = a.n;
    const int r0 = (int)(pix / a.cols), c0 = (int)(pix % a.cols);
    const uint32_t* wt = a.wts + pix * a.nul;
    if (w == 0) {
        const bool cen = shp_get(wt, shp_flat(0, 0, a.Nx, a.Ny));
        const int cnt = build_position_list<64>(wt, cen, r0, c0, a.rows, a.cols, a.Nx, a.Ny, lane, list);
        if (lane < 16) list[cnt + lane] = -1;
        if (lane == 0) L.cnt = cen ? cnt : -1;
    }
    __syncthreads();
    const int K = __builtin_amdgcn_readfirstlane(L.cnt);
    if (K < 0 || K < a.min_nb) {
        __syncthreads();
        return -1;
    }
    const int i = lane & 15, q = lane >> 4;
    const int date = 16 * w + i;
    const float2* band = a.slc + (long long)(date < n ? date : 0) * a.npx;
    mf64x4 R[T == 2 ? 3 : T], I[T == 2 ? 3 : T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) R[t][r] = I[t][r] = 0.0;
    // the last tile of an even NW is its partner wave's too
    const int tiles = NW % 2 == 0 && NW > 1 && w >= NW / 2 ? T - 1 : T;
    float2 f[4];
    auto fetch = [&](int base) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int pos = base < K ? list[base + 4 * s + q] : -1;
            f[s] = make_float2(0.0f, 0.0f);
            if (pos >= 0 && date < n) f[s] = band[pos];
        }
    };
    fetch(0);
    int buf = 0;
    for (int base = 0; base < K; base += 16) {
        float2(*z)[LdsGram64<NW>::S] = L.z[buf];
        buf ^= 1;   // alternate buffers: one barrier per 16 positions
#pragma unroll
        for (int s = 0; s < 4; ++s) z[4 * s + q][date] = f[s];
        __syncthreads();
        if (base + 16 < K) fetch(base + 16);
        // 16 positions are summed by themselves and then added: one long chain
        // of additions through the matrix unit lost more (8.6e-16 of the
        // coherence against 3.2e-16 on the vector unit)
        mf64x4 r[T == 2 ? 3 : T], m[T == 2 ? 3 : T];
#pragma unroll
        for (int t = 0; t < T; ++t) r[t] = m[t] = mf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (base + 4 * s >= K) continue;
            const float2 u = z[4 * s + q][16 * w + i];
            const double ar = (double)u.x, ai = (double)u.y, nar = -(double)u.x;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (t >= tiles) continue;
                double br = ar, bi = ai;
                if (t > 0) {
                    const int J = w + t >= NW ? w + t - NW : w + t;
                    const float2 v = z[4 * s + q][16 * J + i];
                    br = (double)v.x;
                    bi = (double)v.y;
                }
                r[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, r[t], 0, 0, 0);
                m[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, m[t], 0, 0, 0);
                r[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, bi, r[t], 0, 0, 0);
                m[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(nar, bi, m[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < T; ++t)
            if (t < tiles) {
                R[t] += r[t];
                I[t] += m[t];
            }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (i == 4 * r + q) L.dg[date] = R[0][r];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (t >= tiles) continue;
        const int J = w + t >= NW ? w + t - NW : w + t;
        const int col = 16 * J + i;
        const double dc = L.dg[col];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * w + 4 * r + q;
            // Gamma_ij = sum z_i conj(z_j) / sqrt(D_i D_j) (evd.cpp:573-579)
            const double x = L.dg[row] * dc;
            double s = __builtin_amdgcn_rsq(x);
            s = s * fma(-0.5 * x * s, s, 1.5);
            s = s * fma(-0.5 * x * s, s, 1.5);
            // rounded as a quotient by the rounded root is
            double root = x * s;
            root = fma(fma(-root, root, x), 0.5 * s, root);
            double gr = R[t][r] * s, gi = I[t][r] * s;
            gr = fma(fma(-gr, root, R[t][r]), s, gr);
            gi = fma(fma(-gi, root, I[t][r]), s, gi);
            if (row < n && col < n) {
                if (t == 0) {   // the diagonal tile: its upper triangle and the mirror
                    if (col == row) gam[(size_t)row * n + row] = cx<double>{1.0, 0.0};
                    if (col > row) {
                        gam[(size_t)row * n + col] = cx<double>{gr, gi};
                        gam[(size_t)col * n + row] = cx<double>{gr, -gi};
                    }
                } else {
                    gam[(size_t)row * n + col] = cx<double>{gr, gi};
                    gam[(size_t)col * n + row] = cx<double>{gr, -gi};
                }
            }
        }
    }
    __syncthreads();   // list and L are free again
    return K;
}

}  // namespace fringe
