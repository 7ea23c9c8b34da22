// solve_mfma_wg.hpp -- the matrix-core estimator chain of solve_mfma.hpp for
// 33 to 128 dates: one pixel per workgroup of NT = 2, 3 or 4 waves, wave w
// holding rows 32 w .. 32 w + 31 of every matrix as NT accumulator tiles.
//
// A pivot row of the FP32 sweep (and a panel of four pivot rows of the FP64
// one) is published in LDS by the wave that holds it, one barrier a pivot;
// every wave then updates its own tiles, 2 NT MFMAs (32x32x2) a pivot and
// 4 NT (16x16x4) a panel.  Products with the explicit inverse add the waves'
// partial sums through LDS; every wave keeps the whole vector, so norms,
// shifts and the certification run alike in all of them without exchange.
//
// Bound by the matrix instructions and the vector unit together (65-95 % of
// the kernel's cycles; the rest is the latency of a pivot's chain).  Solve
// stage against the register-row and one-row-per-lane solvers it replaced:
// 48 dates (208 x 224, EMI) 4.8 -> 2.8 ms, 64 dates (131 k pixels, EVD) 15.1
// -> 3.9 ms, 96 dates (256 x 256, EMI) 37.4 -> 21.1 ms, with the pixels left
// to the FP64 re-solve down from 10.9 k, 0 and 38.5 k to 4.4 k, 0 and 19.5 k.
// (Before refine_wg 2.6, 3.6 and 21.0 ms, and errors of kept pixels beyond
// the certificate's estimate.)
#pragma once
#include "solve_mfma.hpp"

namespace fringe {

// The wave's accumulator tiles (two tiles padded to three: the compiler turns
// an array of two into one 32-element vector, which it then copies on every
// pivot; the third is never used).
template <int NT> using Tiles = mf32x16[NT == 2 ? 3 : NT];

template <int NT, bool INV> struct LdsMfmaWg {
    static constexpr int N = 32 * NT, S = N + 4;
    float T[INV ? N * S : 4];            // |Gamma|^-1, row-major
    union {
        float row[2][NT][64];            // pivot row: (re | im) per 32 columns
        double panel[2][2 * NT][64];     // four rows of |Gamma|: B operands of 16 columns
        cx<float> part[2][NT][N];        // the waves' partial products
    };
    float xr[NT][32], xi[NT][32];
    double red[2][NT][2];
};

// Sum of x (alike in the wave's lanes) over the workgroup's waves.
template <int NT, bool INV>
__device__ __forceinline__ float wg_sum(LdsMfmaWg<NT, INV>& L, int w, int& turn, float x) {
    turn ^= 1;
    if (lane_now() == 0) L.red[turn][w][0] = (double)x;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < NT; ++k) s += (float)L.red[turn][k][0];
    return uni(s);
}

// Complex sweep of pivots 0 .. n - 1 (as sweep32): the wave's rows of
// (R, I) become those of -B^-1 + I.
template <int NT, bool INV>
__device__ __forceinline__ void sweep_wg(LdsMfmaWg<NT, INV>& L, Tiles<NT>& R, Tiles<NT>& I, int n, int w,
                                         int lane, int& neg, int& near) {
    neg = 0;
    near = 0x7fffffff;
    const uint32_t flip = lane < 32 ? 0u : 0x80000000u;
    int turn = 0;      // one barrier a pivot: consecutive pivots take alternate buffers
    __syncthreads();   // the buffers' last use is over
    for (int K = 0; K < NT; ++K) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = 8 * (v / 4) + 4 * h + v % 4;
                if (32 * K + j < fresh(n)) {
                    float(*row)[64] = L.row[turn];
                    turn ^= 1;
                    if (w == K) {
#pragma unroll
                        for (int J = 0; J < NT; ++J) {
                            float b[2];
                            swap32(R[J][v], I[J][v], b[0], b[1]);
                            row[J][lane] = b[h];
                        }
                    }
                    __syncthreads();
                    const int pb = __builtin_amdgcn_readfirstlane(__float_as_int(row[K][j]));
                    float b[NT], c[NT];
                    const float own = row[w][lane];
#pragma unroll
                    for (int J = 0; J < NT; ++J) {
                        b[J] = row[J][lane];
                        c[J] = row[J][lane ^ 32];
                    }
                    neg += (uint32_t)pb < 0xBF800000u ? 0 : 1;
                    near = min(near, abs(pb - (int)0xBF800000));
                    const float q = -__builtin_amdgcn_rcpf(__int_as_float(pb) + 1.0f);
                    const float a = own * q;
                    const float d = __uint_as_float(__float_as_uint(a) ^ flip);
#pragma unroll
                    for (int J = 0; J < NT; ++J) {
                        R[J] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b[J], R[J], 0, 0, 0);
                        I[J] = __builtin_amdgcn_mfma_f32_32x32x2f32(d, c[J], I[J], 0, 0, 0);
                    }
                }
            }
    }
    __syncthreads();
}

// y = M x: x and y are held whole by every wave, component 32 J + col of J.
template <int NT, bool INV>
__device__ __forceinline__ void apply_wg(LdsMfmaWg<NT, INV>& L, const Tiles<NT>& R, const Tiles<NT>& I,
                                         const cx<float> (&x)[NT], cx<float> (&y)[NT], int w, int col, int h,
                                         int& turn) {
#pragma unroll
    for (int J = 0; J < NT; ++J)
        if (J == w && h == 0) {
            L.xr[w][col] = x[J].re;
            L.xi[w][col] = x[J].im;
        }
    wsync();
    turn ^= 1;
    float re[NT], im[NT];
#pragma unroll
    for (int J = 0; J < NT; ++J) re[J] = im[J] = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {   // four rows at a time
        const float4 p = *(const float4*)&L.xr[w][8 * q + 4 * h];
        const float4 s = *(const float4*)&L.xi[w][8 * q + 4 * h];
        const float xr[4] = {p.x, p.y, p.z, p.w}, xi[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int J = 0; J < NT; ++J) {   // conj(M_rc) x_r
                const int v = 4 * q + k;
                re[J] = fmaf(R[J][v], xr[k], re[J]);
                im[J] = fmaf(R[J][v], xi[k], im[J]);
                re[J] = fmaf(I[J][v], xi[k], re[J]);
                im[J] = fmaf(-I[J][v], xr[k], im[J]);
            }
    }
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        const cx<float> s = {both32(re[J]), both32(im[J])};
        if (h == 0) L.part[turn][w][32 * J + col] = s;
    }
    __syncthreads();
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        y[J] = L.part[turn][0][32 * J + col];
#pragma unroll
        for (int k = 1; k < NT; ++k) y[J] = cadd(y[J], L.part[turn][k][32 * J + col]);
    }
}

template <int NT> struct EigStateWg {
    cx<float> x[NT];
    float theta, dn, q, dq;
    bool done;
};

template <int NT> __device__ __forceinline__ float norm2_wg(const cx<float> (&x)[NT]) {
    float s = 0.0f;
#pragma unroll
    for (int J = 0; J < NT; ++J) s += cabs2(x[J]);
    return uni(red32<OpAdd>(s));
}

// One normalised step x -> y / (x^H y) (y = B^-1 x, or Gamma x): the Rayleigh
// quotient into E.theta, the squared change returned.
template <int NT>
__device__ __forceinline__ float step_wg(EigStateWg<NT>& E, const cx<float> (&y)[NT]) {
    float t = 0.0f;
#pragma unroll
    for (int J = 0; J < NT; ++J) t = fmaf(y[J].re, E.x[J].re, fmaf(y[J].im, E.x[J].im, t));
    E.theta = uni(red32<OpAdd>(t));
    const float it = __builtin_amdgcn_rcpf(E.theta);
    cx<float> d[NT];
#pragma unroll
    for (int J = 0; J < NT; ++J) d[J] = cx<float>{fmaf(y[J].re, it, -E.x[J].re), fmaf(y[J].im, it, -E.x[J].im)};
    const float d2 = norm2_wg<NT>(d);
    const float s = __builtin_amdgcn_rsqf(1.0f + d2);
#pragma unroll
    for (int J = 0; J < NT; ++J) E.x[J] = cx<float>{(E.x[J].re + d[J].re) * s, (E.x[J].im + d[J].im) * s};
    return d2;
}

// Inverse iteration with B^-1 = I - M, as iterate32.
template <int NT, bool INV>
__device__ __forceinline__ void iterate_wg(LdsMfmaWg<NT, INV>& L, const Tiles<NT>& R, const Tiles<NT>& I, int w,
                                           int col, int h, int& turn, float qb, EigStateWg<NT>& E) {
    float dp = 0.0f;
    const float left = scal(4.0e-7f * (1.0f - qb)), qq = scal(qb * qb);
    if (!(qb > 0.0f)) E.q = E.dq = 0.0f;
    cx<float> y[NT];
    for (int k = qb > 0.0f ? 0 : -2; k < 24; ++k) {
        apply_wg<NT, INV>(L, R, I, E.x, y, w, col, h, turn);
#pragma unroll
        for (int J = 0; J < NT; ++J) y[J] = csub(E.x[J], y[J]);
        if (k < 0) {   // plain products first: the start vector is far off
            const float nr = k < -1 ? 1.0f : __builtin_amdgcn_rsqf(norm2_wg<NT>(y));
#pragma unroll
            for (int J = 0; J < NT; ++J) E.x[J] = cscale(y[J], nr);
            continue;
        }
        const float dn = __builtin_amdgcn_sqrtf(step_wg<NT>(E, y));
        E.dn = dn;
        E.done = false;
        if (!(dn < 3.0e38f)) return;   // not finite
        if (qb > 0.0f) {
            E.done = dn * qq < left;
            if (E.done) return;
            continue;
        }
        if (dn < 4.0e-7f) E.done = true;
        if (k > 0) {
            E.q = dn * __builtin_amdgcn_rcpf(dp);
            E.dq = dn;
            const float q = fminf(E.q, 0.99f);
            if (dn * q * q < 4.0e-7f * (1.0f - q)) E.done = true;
            if (k > 1 && E.q > kSlow && dn > 2.0e-5f && !E.done) return;
        }
        if (E.done) return;
        dp = dn;
    }
}

// FP64 sweep of |Gamma| by panels of four pivots (diagonal stored minus 1,
// padding as in sweep64): the wave's rows become those of -|Gamma|^-1 + I.
// The 4 x 4 pivot block is inverted by 2 x 2 blocks, alike in every lane; each
// lane picks its entry of the inverse as the A operand of the 4x4x4 MFMA.
template <int NT, bool INV>
__device__ __forceinline__ bool sweep64_wg(LdsMfmaWg<NT, INV>& L, mf64x4 (&M)[2][2 * NT], int n, int w, int lane,
                                           bool& near) {
    bool ok = true;
    near = false;
    const int i = lane & 3, q = lane >> 4;
    int turn = 0;
    __syncthreads();   // the buffers' last use is over
    for (int K = 0; K < NT; ++K) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (32 * K + 16 * kk + 4 * r < fresh(n) && ok) {
                    double(*X)[64] = L.panel[turn];
                    turn ^= 1;
                    if (w == K) {
#pragma unroll
                        for (int J = 0; J < 2 * NT; ++J) X[J][lane] = M[kk][J][r];
                    }
                    __syncthreads();
                    const double* D = &X[2 * K + kk][4 * r];   // D[q][t] at 16 q + t
                    const double a00 = D[0] + 1.0, a01 = D[1], a11 = D[17] + 1.0;
                    const double b00 = D[2], b01 = D[3], b10 = D[18], b11 = D[19];
                    const double c00 = D[34] + 1.0, c01 = D[35], c11 = D[51] + 1.0;
                    // A^-1
                    const double da = fma(-a01, a01, a00 * a11), ra = fast_rcp(da);
                    const double e00 = a11 * ra, e01 = -a01 * ra, e11 = a00 * ra;
                    // T = A^-1 B, S = C - B^T T
                    const double t00 = fma(e00, b00, e01 * b10), t01 = fma(e00, b01, e01 * b11);
                    const double t10 = fma(e01, b00, e11 * b10), t11 = fma(e01, b01, e11 * b11);
                    const double s00 = fma(-b00, t00, fma(-b10, t10, c00));
                    const double s01 = fma(-b00, t01, fma(-b10, t11, c01));
                    const double s11 = fma(-b01, t01, fma(-b11, t11, c11));
                    const double ds = fma(-s01, s01, s00 * s11), rs = fast_rcp(ds);
                    if (!(fmin(da, a00 * a00) >= kCertPivotMin * a00) || !(a00 > 0.0) ||
                        !(fmin(ds, s00 * s00) >= kCertPivotMin * s00) || !(s00 > 0.0)) {   // rarely
                        near = near | (fabs(a00) < kCertPivotMin) | (fabs(da) < kCertPivotMin * a00);
                        ok = (a00 > 0.0) & (da > 0.0);
                        if (ok) {
                            near = near | (fabs(s00) < kCertPivotMin) | (fabs(ds) < kCertPivotMin * s00);
                            ok = (s00 > 0.0) & (ds > 0.0);
                        }
                    }
                    // the inverse, negated: [A^-1 + T S^-1 T^T, -T S^-1; ., S^-1]
                    const double f00 = s11 * rs, f01 = -s01 * rs, f11 = s00 * rs;
                    const double g00 = fma(t00, f00, t01 * f01), g01 = fma(t00, f01, t01 * f11);
                    const double g10 = fma(t10, f00, t11 * f01), g11 = fma(t10, f01, t11 * f11);
                    const double h00 = fma(g00, t00, fma(g01, t01, e00));
                    const double h01 = fma(g00, t10, fma(g01, t11, e01));
                    const double h11 = fma(g10, t10, fma(g11, t11, e11));
                    const bool i0 = (i & 1) == 0, q0 = (q & 1) == 0;
                    const double tl = i0 ? (q0 ? h00 : h01) : (q0 ? h01 : h11);
                    const double br = i0 ? (q0 ? f00 : f01) : (q0 ? f01 : f11);
                    const double tr = i0 ? (q0 ? g00 : g01) : (q0 ? g10 : g11);   // row i < 2, column q >= 2
                    const double bl = q0 ? (i0 ? g00 : g01) : (i0 ? g10 : g11);   // its transpose
                    const double ca = i < 2 ? (q < 2 ? -tl : tr) : (q < 2 ? bl : -br);
                    double b[2 * NT], wv[2];
#pragma unroll
                    for (int J = 0; J < 2 * NT; ++J) b[J] = X[J][lane];
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        wv[k] = __builtin_amdgcn_mfma_f64_4x4x4f64(ca, X[2 * w + k][lane], 0.0, 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int J = 0; J < 2 * NT; ++J)
                            M[k][J] = __builtin_amdgcn_mfma_f64_16x16x4f64(wv[k], b[J], M[k][J], 0, 0, 0);
                }
            }
    }
    __syncthreads();
    return ok;
}

// Above 96 dates a wave's tiles leave few registers: loads of one tile at a
// time are in flight (all of them at once spilled).
template <int NT> __device__ __forceinline__ void tile_fence_wg() {
    if constexpr (NT >= 4) __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void load_tile_wg(const GammaBuf& gam, int n, int w, int J, int col, int h, mf32x16& R,
                                             mf32x16& I) {
    int o = fresh_lane(gam.offset(32 * w + 4 * h, 32 * J + col));
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const cx<float> g = gam.at(o);
        o += (v % 4 == 3 ? 5 : 1) * n * 8;
        R[v] = g.re;
        I[v] = g.im;
    }
}

template <int NT>
__device__ __forceinline__ void load_gamma_wg(const GammaBuf& gam, int n, int w, int col, int h, Tiles<NT>& R, Tiles<NT>& I) {
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        load_tile_wg(gam, n, w, J, col, h, R[J], I[J]);
        tile_fence_wg<NT>();
    }
}

// Register of tile (w, w)'s diagonal in this lane, or -1.
__device__ __forceinline__ int diagonal_wg(int col, int h) {
    return ((col >> 2) & 1) == h ? 4 * (col >> 3) + (col & 3) : -1;
}

// The step in residual form, as refine32; A = T o Gamma (INV) or Gamma.
template <int NT, bool INV>
__device__ __forceinline__ float refine_wg(LdsMfmaWg<NT, INV>& L, const GammaBuf& gam, const Tiles<NT>& R,
                                          const Tiles<NT>& I, int n, int w, int band, float sg, int& turn,
                                          EigStateWg<NT>& E) {
    const int lane = lane_now(), col = lane & 31, h = lane >> 5;
#pragma unroll
    for (int J = 0; J < NT; ++J)
        if (J == w && h == 0) {
            L.xr[w][col] = E.x[J].re;
            L.xi[w][col] = E.x[J].im;
        }
    wsync();
    turn ^= 1;
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        int o = fresh_lane(gam.offset(32 * w + 4 * h, 32 * J + col));
        const int d0 = fresh_lane(col - 4 * h - 32 * w);
        float re = 0.0f, im = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 xr = *(const float4*)&L.xr[w][8 * q + 4 * h], xi = *(const float4*)&L.xi[w][8 * q + 4 * h];
            const float pr[4] = {xr.x, xr.y, xr.z, xr.w}, pi[4] = {xi.x, xi.y, xi.z, xi.w};
            float m[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            if constexpr (INV) {
                const float4 t = *(const float4*)&L.T[(32 * J + col) * LdsMfmaWg<NT, INV>::S + 32 * w + 8 * q + 4 * h];
                m[0] = t.x; m[1] = t.y; m[2] = t.z; m[3] = t.w;
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const cx<float> g = gam.at(o);
                o += (b == 3 ? 5 : 1) * n * 8;
                const bool out = !INV && band > 0 && abs(8 * q + b - d0 - 32 * J) > band;
                const float ar = out ? 0.0f : g.re * m[b], ai = out ? 0.0f : g.im * m[b];
                re = fmaf(ar, pr[b], re);
                im = fmaf(ar, pi[b], im);
                re = fmaf(ai, pi[b], re);
                im = fmaf(-ai, pr[b], im);
            }
            __builtin_amdgcn_sched_barrier(0);   // four rows' loads in flight (more of them spilled)
        }
        const cx<float> s = {both32(re), both32(im)};
        if (h == 0) L.part[turn][w][32 * J + col] = s;
    }
    __syncthreads();
    cx<float> r[NT], z[NT];
    float t = 0.0f;
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        r[J] = L.part[turn][0][32 * J + col];
#pragma unroll
        for (int k = 1; k < NT; ++k) r[J] = cadd(r[J], L.part[turn][k][32 * J + col]);
        t = fmaf(r[J].re, E.x[J].re, fmaf(r[J].im, E.x[J].im, t));
    }
    t = uni(red32<OpAdd>(t));
#pragma unroll
    for (int J = 0; J < NT; ++J) r[J] = cx<float>{fmaf(-t, E.x[J].re, r[J].re), fmaf(-t, E.x[J].im, r[J].im)};
    apply_wg<NT, INV>(L, R, I, r, z, w, col, h, turn);
    float cr = 0.0f, ci = 0.0f;   // along x the change means nothing
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        z[J] = csub(r[J], z[J]);
        cr = fmaf(E.x[J].re, z[J].re, fmaf(E.x[J].im, z[J].im, cr));
        ci = fmaf(E.x[J].re, z[J].im, fmaf(-E.x[J].im, z[J].re, ci));
    }
    cr = uni(red32<OpAdd>(cr));
    ci = uni(red32<OpAdd>(ci));
#pragma unroll
    for (int J = 0; J < NT; ++J)
        z[J] = cx<float>{fmaf(-cr, E.x[J].re, fmaf(ci, E.x[J].im, z[J].re)),
                         fmaf(-cr, E.x[J].im, fmaf(-ci, E.x[J].re, z[J].im))};
    const float d2 = norm2_wg<NT>(z), s = __builtin_amdgcn_rsqf(1.0f + d2);
#pragma unroll
    for (int J = 0; J < NT; ++J) E.x[J] = cx<float>{fmaf(-sg, z[J].re, E.x[J].re) * s, fmaf(-sg, z[J].im, E.x[J].im) * s};
    return d2;
}

// One pixel on the NT waves of a workgroup.
template <int MODE, int NT>
__device__ __forceinline__ void solve_mfma_wg_pixel(const SolveArgs& a, LdsMfmaWg<NT, MODE != MODE_EVD>& L, int w,
                                                    int np, const GammaBuf& gam, long long pix) {
    constexpr bool INV = MODE != MODE_EVD;
    constexpr int S = LdsMfmaWg<NT, INV>::S;
    const int n = a.n;
    const bool stbas = a.method == FRINGE_METHOD_STBAS && MODE == MODE_EVD;
    float code = 0.0f;
    bool unc = false;
    bool inv = INV;
    int turn = 0;
    EigStateWg<NT> E;

    const bool act = np >= 0;
    // What follows from the lane is computed again in each stage: held over
    // the sweeps it spilled.
    if (act) {
        const int lane = lane_now(), col = lane & 31, h = lane >> 5;
        if constexpr (MODE == MODE_MLE) {
            const int vd0 = diagonal_wg(col, h);
            Tiles<NT> R, I;
            load_gamma_wg<NT>(gam, n, w, col, h, R, I);
            const float s = 1.0e-6f + kCertThrMargin * Lim<float>::eps() * (float)n;
            float sum = 0.0f;
#pragma unroll
            for (int J = 0; J < NT; ++J)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    sum += fabsf(R[J][v]) + fabsf(I[J][v]);
                    if (J == w && v == vd0) R[J][v] = -s;
                }
            sum = wg_sum(L, w, turn, __all(sum < 3.0e38f) ? 0.0f : 1.0f);
            if (sum > 0.0f) {
                code = -1.0f;
            } else {
                int neg, near;
                sweep_wg<NT, INV>(L, R, I, n, w, lane, neg, near);
                unc = neg != 0;
            }
        }
        if constexpr (INV) {
            if (code == 0.0f && !unc) {
                mf64x4 M[2][2 * NT];
                float sum = 0.0f;
                const int rb = 32 * w + (lane >> 4);
#pragma unroll
                for (int J = 0; J < 2 * NT; ++J) {
                    int o = fresh_lane(gam.offset(rb, 16 * J + (lane & 15)));
                    const int dr = 16 * J + (lane & 15) - rb;   // 16 k + 4 r on the diagonal
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const cx<float> g = gam.at(o);
                            o += 4 * n * 8;
                            float v = __builtin_amdgcn_sqrtf(g.re * g.re + g.im * g.im);
                            if (dr == 16 * k + 4 * r) v = 0.0f;
                            sum += v;
                            M[k][J][r] = (double)v;
                        }
                    tile_fence_wg<NT>();
                }
                sum = wg_sum(L, w, turn, __all(sum < 3.0e38f) ? 0.0f : 1.0f);
                if (sum > 0.0f) {
                    code = -1.0f;
                } else {
                    bool near;
                    const bool pd = sweep64_wg<NT, INV>(L, M, n, w, lane, near);
                    unc = near;
                    if (MODE == MODE_EMI) inv = pd;
                    else unc = unc || !pd;
                    if (inv) {
#pragma unroll
                        for (int J = 0; J < 2 * NT; ++J)
#pragma unroll
                            for (int k = 0; k < 2; ++k)
#pragma unroll
                                for (int r = 0; r < 4; ++r) {
                                    const int row = rb + 16 * k + 4 * r, c = 16 * J + (lane & 15);
                                    L.T[row * S + c] = (float)((row == c ? 1.0 : 0.0) - M[k][J][r]);
                                }
                    }
                    __syncthreads();
                    if constexpr (MODE == MODE_MLE) {
                        float tr = 0.0f;
#pragma unroll
                        for (int J = 0; J < NT; ++J)
                            if (32 * J + col < n) tr += L.T[(32 * J + col) * (S + 1)];
                        unc = unc || !(uni(red32<OpAdd>(tr)) < 1.0e5f);
                    }
                }
            }
        }
    }

    // ---- the eigenpair ----
    if (act && code == 0.0f && !unc) {
        float sigma = 1.0f, sg = 1.0f, tn = 1.0f;
        {
        const int lane = lane_now(), col = lane & 31, h = lane >> 5;
        const float is = __builtin_amdgcn_rsqf((float)n);
#pragma unroll
        for (int J = 0; J < NT; ++J) {   // start: the phases of the middle column
            const bool in = 32 * J + col < n;
            const cx<float> g = gam.at(gam.offset(n >> 1, 32 * J + col));
            const float g2 = cabs2(g);
            const float s = g2 > 0.0f ? __builtin_amdgcn_rsqf(g2) * is : 0.0f;
            E.x[J] = cx<float>{g.re * s, -g.im * s};
            if (in && !(g2 > 0.0f)) E.x[J].re = is;
        }
        if (!inv) {
            sg = -1.0f;
            if constexpr (INV) {   // EMI's fallback: Gamma = T o Gamma (read behind the sum's barrier)
                for (int e = threadIdx.x; e < LdsMfmaWg<NT, INV>::N * S; e += 64 * NT) L.T[e] = 1.0f;
            }
            Tiles<NT> R, I;
            load_gamma_wg<NT>(gam, n, w, col, h, R, I);
            const int d0 = col - 4 * h - 32 * w;   // column - row of register 0 of tile 0
            float f2 = 0.0f;
#pragma unroll
            for (int J = 0; J < NT; ++J)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if (stbas && abs(8 * (v / 4) + v % 4 - d0 - 32 * J) > a.bw) {
                        R[J][v] = 0.0f;
                        I[J][v] = 0.0f;
                    }
                    f2 = fmaf(R[J][v], R[J][v], fmaf(I[J][v], I[J][v], f2));
                }
            f2 = wg_sum(L, w, turn, uni(both32(red32<OpAdd>(f2))));
            if (MODE == MODE_EVD && !(f2 < 3.0e38f)) code = -6.0f;
            if (code == 0.0f) {
                float d2 = 1.0f;
                cx<float> y[NT];
                for (int k = 0; k < 4; ++k) {
                    apply_wg<NT, INV>(L, R, I, E.x, y, w, col, h, turn);
                    d2 = step_wg<NT>(E, y);
                }
                sigma = E.theta + E.theta * fmaxf(__builtin_amdgcn_sqrtf(d2), 0.02f);
                sigma = scal(sigma);
                tn = scal(1.0f + __builtin_amdgcn_sqrtf(fmaxf(f2 * a.inv_n - 1.0f, 0.0f) * (float)(fresh(n) - 1)));
            }
        }
        }
        bool certified = false, checking = false, close = false;
        float lam = 0.0f, delta = 0.0f;
        if (code == 0.0f)
            for (int att = 0; att < 6; ++att) {
                const int lane = lane_now(), col = lane & 31, h = lane >> 5;
                const int vd = diagonal_wg(col, h), d0 = col - 4 * h - 32 * w;
                // ---- B = +-(A - sigma I), diagonal minus 1 ----
                const int own = 32 * w + col;
                const float dg = inv ? (own < n ? L.T[own * (S + 1)] : 0.0f) : 1.0f;
                const float off = own < n ? sg * (dg - sigma) - 1.0f : 0.0f;
                Tiles<NT> R, I;
                if (inv) {
                    float f2 = 0.0f;
#pragma unroll
                    for (int J = 0; J < NT; ++J) {
                        load_tile_wg(gam, n, w, J, col, h, R[J], I[J]);
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float4 m = *(const float4*)&L.T[(32 * J + col) * S + 32 * w + 8 * q + 4 * h];
                            const float mm[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
                            for (int b = 0; b < 4; ++b) {
                                const int v = 4 * q + b;
                                R[J][v] *= mm[b];
                                I[J][v] *= mm[b];
                                f2 = fmaf(R[J][v], R[J][v], fmaf(I[J][v], I[J][v], f2));
                                if (J == w && v == vd) R[J][v] = off;
                            }
                        }
                        tile_fence_wg<NT>();
                    }
                    if (att == 0) {   // |H| <= m + s sqrt(n - 1), as in solve_mfma_pixel
                        float tr = 0.0f;
#pragma unroll
                        for (int J = 0; J < NT; ++J)
                            if (32 * J + col < n) tr += L.T[(32 * J + col) * (S + 1)];
                        tr = uni(red32<OpAdd>(tr)) * a.inv_n;
                        const float ff = wg_sum(L, w, turn, uni(both32(red32<OpAdd>(f2)))) * a.inv_n;
                        tn = scal(tr + __builtin_amdgcn_sqrtf(fmaxf(ff - tr * tr, 0.0f) * (float)(fresh(n) - 1)));
                        if (!(tn < 3.0e38f)) break;
                    }
                } else {
#pragma unroll
                    for (int J = 0; J < NT; ++J) {
                        load_tile_wg(gam, n, w, J, col, h, R[J], I[J]);
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const bool out = stbas && abs(8 * (v / 4) + v % 4 - d0 - 32 * J) > a.bw;
                            R[J][v] = out ? 0.0f : -R[J][v];
                            I[J][v] = out ? 0.0f : -I[J][v];
                            if (J == w && v == vd) R[J][v] = off;
                        }
                        tile_fence_wg<NT>();
                    }
                }
                // the vector waits in LDS (behind the sweep's barriers) for the
                // registers that the sweep needs
#pragma unroll
                for (int J = 0; J < NT; ++J)
                    if (J == w && h == 0) {
                        L.xr[w][col] = E.x[J].re;
                        L.xi[w][col] = E.x[J].im;
                    }
                int neg, near;
                sweep_wg<NT, INV>(L, R, I, n, w, lane, neg, near);
#pragma unroll
                for (int J = 0; J < NT; ++J) E.x[J] = cx<float>{L.xr[J][col], L.xi[J][col]};
                if (checking) {
                    certified = neg <= 1 && near >= 1700;
                    __syncthreads();   // the outputs take the vector's place
                    break;
                }
                if (neg > 1) {
                    if (inv) sigma = sigma > 0.5f ? 0.5f * sigma : 0.0f;
                    else sigma = sigma * 1.15f;
                    sigma = scal(sigma);
                    continue;
                }
                iterate_wg<NT, INV>(L, R, I, w, col, h, turn, 0.0f, E);
                const float mu = scal(__builtin_amdgcn_rcpf(E.theta));
                lam = scal(sigma + sg * mu);
                if (!(fabsf(lam) < 3.0e38f)) break;
                if (!E.done) {
                    const float q = E.q > 0.0f ? fminf(fmaxf(E.q, 1.0e-3f), 0.98f) : 0.98f;
                    const float gap = fabsf(mu) / q - mu;
                    const float e = fminf(E.dn * q / (1.0f - q), 1.0f);
                    sigma = scal(sigma + sg * (mu - (e * e + 0.15f) * gap));
                    continue;
                }
                // ---- certification ----
                float m2 = lit(3.0e38f);   // smallest component
#pragma unroll
                for (int J = 0; J < NT; ++J)
                    if (32 * J + col < n) m2 = fminf(m2, cabs2(E.x[J]));
                m2 = scal(red32<OpMin>(m2));
                delta = scal(cert_eps(inv, a.cert_h, a.cert_g, tn) * (tn * __builtin_amdgcn_rsqf(m2)));
                if (!(delta <= tn)) break;
                float f = 0.0f;
#pragma unroll
                for (int J = 0; J < NT; ++J)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const float x = J == w && v == vd ? 1.0f - R[J][v] : R[J][v];
                        f = fmaf(x, x, fmaf(I[J][v], I[J][v], f));
                    }
                if (vd >= 0 && own >= n) f -= 1.0f;   // padding: R = 0 on the diagonal
                f = wg_sum(L, w, turn, uni(both32(red32<OpAdd>(f))));
                const float s2 = scal(fmaxf(f - E.theta * E.theta, 0.0f) + 4.0e-6f * f), t = scal(mu + delta);
                const bool side = neg == 0 ? E.theta > 0.0f : E.theta < 0.0f;
                if (!side) break;
                // the contraction is at most qb: the error left by the last step
                const float qb = scal(__builtin_amdgcn_sqrtf(s2) * fabsf(mu));
                bool conv = qb < 0.8f;
                if (conv && E.dn * qb * qb > 4.0e-7f * (1.0f - qb)) {
                    iterate_wg<NT, INV>(L, R, I, w, col, h, turn, qb, E);
                    conv = E.done;
                }
                // a shift inside the spectrum: small pivots would have cost accuracy
                if (neg != 0 && near < kNearInside && !close) conv = false;
                certified = conv && (t <= 0.0f || s2 * t * t < 1.0f);
                if (certified || (conv && close)) {
                    const float most = scal(refined2(m2, qb, tn * fabsf(E.theta)));
                    float d2 = 1.0f;
                    for (int k = 0; k < kRefines && d2 > most; ++k)
                        d2 = scal(refine_wg<NT, INV>(L, gam, R, I, fresh(n), w, stbas ? a.bw : 0, sg, turn, E));
                    if (!(d2 <= most)) certified = conv = false;
                }
                if (certified) break;
                // the next eigenvalue as the measured contraction places it is
                // too close for any certificate: the FP64 path's pixel
                if (E.q > 0.02f && E.dq > 4.0e-6f && fabsf(mu) * __builtin_amdgcn_rcpf(E.q) - mu < 0.7f * delta) break;
                if (!close) {   // once more from a quarter of the distance away
                    close = true;
                    sigma = scal(lam - sg * (0.25f * delta));
                    continue;
                }
                if (!conv) break;
                checking = true;
                sigma = scal(lam + sg * delta);
            }
        if constexpr (MODE != MODE_EMI) unc = unc || !(lam >= 1.0e-6f + kCertThrMargin * Lim<float>::eps() * tn);
        unc = code == 0.0f && (unc || !certified);
    }

    const int lane = lane_now(), col = lane & 31, h = lane >> 5;
    if (act && unc) {   // the FP64 re-solve writes every output of the pixel
        if (w == 0 && lane == 0) {
            const int e = atomicAdd(a.cert_count, 1);
            if (e < a.cert_cap) a.cert_list[e] = (int)pix;
        }
        return;
    }
    const int date = 32 * w + col;   // of the wave's share of the outputs
    if (!act || code != 0.0f) {
        if (h == 0 && date < n) a.phase[(long long)date * a.npx + pix] = make_float2(0.0f, 0.0f);
        if (w == 0 && lane == 0) {
            a.tcorr[pix] = act ? code : 0.0f;
            a.comp[pix] = make_float2(0.0f, 0.0f);
        }
        return;
    }

    // ---- referenced phases (evd.cpp:738-749) ----
    cx<float> vref = {0.0f, 0.0f};
#pragma unroll
    for (int J = 0; J < NT; ++J)
        if (J == a.ref / 32) vref = cx<float>{lane_f32(E.x[J].re, a.ref & 31), lane_f32(E.x[J].im, a.ref & 31)};
    cx<float> o[NT];
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        const cx<float> uv = cmulc(E.x[J], vref);
        const float u2 = cabs2(uv);
        float ur = __builtin_amdgcn_rsqf(u2);
        ur = ur * fmaf(-0.5f * u2 * ur, ur, 1.5f);   // one Newton step
        o[J] = cscale(uv, ur);
        if (__any(32 * J + col < n && !(u2 > 1.0e-36f))) {   // a zero, or nearly, component
            bool okr, oku, okv;
            const cx<float> cref = unit_or(cconj(vref), cx<float>{1.0f, 0.0f}, okr);
            const cx<float> u = unit_or(uv, cx<float>{0.0f, 0.0f}, oku);
            o[J] = oku ? u : (okr ? cref : unit_or(E.x[J], cx<float>{1.0f, 0.0f}, okv));
        }
        if (32 * J + col == a.ref) o[J] = cx<float>{1.0f, 0.0f};
    }
    // ---- compressed SLC (evd.cpp:755-762) ----
    cx<double> cs = {0.0, 0.0};
#pragma unroll
    for (int J = 0; J < NT; ++J)
        if (J == w) {
            if (h == 0) {
                if (date < n) a.phase[(long long)date * a.npx + pix] = make_float2(o[J].re, o[J].im);
                L.xr[w][col] = date < n ? o[J].re : 0.0f;
                L.xi[w][col] = date < n ? o[J].im : 0.0f;
            }
            if (date >= a.ref && date < n) {
                const float2 z = a.slc[(long long)date * a.npx + pix];
                cs.re = (double)(z.x * o[J].re + z.y * o[J].im);
                cs.im = (double)(z.y * o[J].re - z.x * o[J].im);
            }
        }
    cs = cx<double>{red32<OpAdd>(cs.re), red32<OpAdd>(cs.im)};
    wsync();
    // ---- temporal coherence (evd.cpp:770-786): the wave's rows against the
    // columns right of them ----
    float xr[16], xi[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 p = *(const float4*)&L.xr[w][8 * q + 4 * h];
        const float4 s = *(const float4*)&L.xi[w][8 * q + 4 * h];
        xr[4 * q] = p.x; xr[4 * q + 1] = p.y; xr[4 * q + 2] = p.z; xr[4 * q + 3] = p.w;
        xi[4 * q] = s.x; xi[4 * q + 1] = s.y; xi[4 * q + 2] = s.z; xi[4 * q + 3] = s.w;
    }
    float sr = 0.0f, si = 0.0f;
#pragma unroll
    for (int J = 0; J < NT; ++J) {
        if (J < w) continue;
        const int c = 32 * J + col;
        const int lo = stbas ? c - a.bw : 0;   // rows lo .. c - 1
        int off = fresh_lane(gam.offset(32 * w + 4 * h, c));
        const int r0 = c - 32 * w - 4 * h, r1 = r0 - c + lo;   // rows r1 <= r < r0, from the lane's first
        float tr = 0.0f, ti = 0.0f;
        mf32x16 gr, gi;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int row = 8 * (v / 4) + v % 4;
            const cx<float> g = gam.at(off);
            off += (v % 4 == 3 ? 5 : 1) * n * 8;
            gr[v] = g.re;
            gi[v] = g.im;
            float rs = __builtin_amdgcn_rsqf(fmaf(g.re, g.re, g.im * g.im));
            rs = row < r0 ? rs : 0.0f;
            if (stbas && row < r1) rs = 0.0f;
            const float pr = g.re * rs, pi = g.im * rs;
            tr = fmaf(pr, xr[v], fmaf(pi, xi[v], tr));
            ti = fmaf(pi, xr[v], fmaf(-pr, xi[v], ti));
        }
        if (__any(c < n && !(fabsf(tr) < 3.0e38f))) {   // a zero entry, whose phase counts as 0
            tr = 0.0f;
            ti = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = 8 * (v / 4) + v % 4;
                const float g2 = fmaf(gr[v], gr[v], gi[v] * gi[v]);
                const bool use = row < r0 && !(stbas && row < r1), z = !(g2 > 0.0f);
                const float rs = use ? __builtin_amdgcn_rsqf(g2) : 0.0f;
                const float pr = z ? (use ? 1.0f : 0.0f) : gr[v] * rs, pi = z ? 0.0f : gi[v] * rs;
                tr = fmaf(pr, xr[v], fmaf(pi, xi[v], tr));
                ti = fmaf(pi, xr[v], fmaf(-pr, xi[v], ti));
            }
        }
        if (c < n) {
            sr = fmaf(tr, o[J].re, fmaf(-ti, o[J].im, sr));
            si = fmaf(tr, o[J].im, fmaf(ti, o[J].re, si));
        }
    }
    sr = uni(both32(red32<OpAdd>(sr)));
    si = uni(both32(red32<OpAdd>(si)));
    sr = wg_sum(L, w, turn, sr);
    si = wg_sum(L, w, turn, si);
    turn ^= 1;
    if (lane == 0) {
        L.red[turn][w][0] = cs.re;
        L.red[turn][w][1] = cs.im;
    }
    __syncthreads();
    if (w == 0 && lane == 0) {
        cx<double> c = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            c.re += L.red[turn][k][0];
            c.im += L.red[turn][k][1];
        }
        const double s2 = (double)sr * (double)sr + (double)si * (double)si;
        double rs = __builtin_amdgcn_rsq(s2);
        rs = rs * fma(-0.5 * s2 * rs, rs, 1.5);
        a.tcorr[pix] = (float)((s2 > 0.0 ? s2 * rs : 0.0) * a.inv_pairs);
        a.comp[pix] = make_float2((float)(c.re * a.inv_comp), (float)(c.im * a.inv_comp));
    }
}

// Waves per SIMD, as many as leave no vector register spilled (the build
// fails on one: a value alike in all lanes, stored to scratch with lanes
// switched off, came back without theirs).  Solve stage with one wave fewer,
// before refine_wg: 64 dates EVD 3.6 -> 4.1 ms, 96 dates EMI 21.0 -> 24.7 ms.
constexpr int waves_wg(int mode, int nt) { return nt == 2 ? (mode == MODE_EVD ? 4 : 3) : nt == 3 && mode != MODE_MLE ? 3 : 2; }
template <int MODE, int NT>
__global__ __launch_bounds__(64 * NT) __attribute__((amdgpu_waves_per_eu(waves_wg(MODE, NT)))) void solve_mfma_wg_kernel(SolveArgs a) {
    __shared__ LdsMfmaWg<NT, MODE != MODE_EVD> L;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slot = a.slots - 1 - (int)blockIdx.x;
    const int np = a.npix[slot];
    const cx<float>* gam = (const cx<float>*)a.gamma + (size_t)slot * a.n * a.n;
    solve_mfma_wg_pixel<MODE, NT>(a, L, w, np, GammaBuf(gam, a.n), a.first + slot);
}

}  // namespace fringe
