// solve_mfma64.hpp -- the FP64 estimator chain on the matrix cores, up to 128
// dates: the plain FP64 path, and the FP64 re-solve of the pixels the mixed
// precisions did not certify (the same code on the same coherence, so that
// the two agree bit for bit).
//
// One pixel per workgroup of NW = ceil(n / 16) waves; wave w holds rows
// 16 w .. 16 w + 15 of every matrix as NW tiles of v_mfma_f64_16x16x4 (lane
// l, register r: column l % 16, row 4 r + l / 16), so that four consecutive
// rows of a tile are one register, laid out as the B operand.  As in
// solve_mfma.hpp, explicit inverses come from the symmetric sweep operator:
// panels of four pivots for the real |Gamma| (one 16x16x4 MFMA a tile), of
// two for the complex B = +-(A - sigma I) (real and imaginary parts fill the
// four k: two MFMAs a tile).  The wave that holds a panel publishes it in
// LDS, one barrier a panel; the pivot block's inverse is applied by a
// v_mfma_f64_4x4x4, which takes and gives the same layout.  Products with the
// inverse use the same instruction, with the vector's real and imaginary
// parts as two rows of A, and add the waves' partial sums through LDS.
//
// There is no other path to leave a pixel to, so the search for the extreme
// eigenpair goes on until the inertia and the Frobenius norm of the inverse
// show that it is the extreme one, or 36 shifts have narrowed it down to a
// cluster of eigenvalues, one of whose vectors is the result.
//
// Bound by the FP64 matrix instructions and, per pivot panel, by the chain
// publish, barrier, read, pivot inverse.  Solve stage against the vector-unit
// solvers it replaced: 301 x 409 pixels of 27 dates (EMI) 4.1 -> 2.5 ms; the
// re-solve with its Gram, a pixel: of 1.1 k pixels of 48 dates 0.74 -> 0.26
// us (0.19 of 4.4 k), of 14.7 k pixels of 96 dates 2.8 -> 1.24 us (1.29 of
// 19.5 k).
#pragma once
#include "gram_mfma64.hpp"

namespace fringe {

template <int NW> struct LdsMfma64 {
    static constexpr int N = 16 * NW;
    union {
        double panel[2][NW][64];        // pivot rows as B operands
        cx<double> part[2][NW][N];      // the waves' partial products
    };
    cx<double> x[NW][16];
    double red[2][NW][2];
};

struct GammaBuf64 {
    __amdgpu_buffer_rsrc_t rsrc;
    int n;
    __device__ __forceinline__ GammaBuf64(const cx<double>* gam, int n_) : n(n_) {
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)gam, 0, n_ * n_ * 16, 0x00027000);
    }
    __device__ __forceinline__ int offset(int row, int c) const { return c < n ? (row * n + c) * 16 : 0x40000000; }
    __device__ __forceinline__ cx<double> at(int off) const {
        const auto u = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
        return cx<double>{__builtin_bit_cast(double, ((uint64_t)u[1] << 32) | u[0]),
                          __builtin_bit_cast(double, ((uint64_t)u[3] << 32) | u[2])};
    }
};

// Tiles of a wave; NW = 2 and 4 padded, as in solve_mfma_wg.hpp.
template <int NW> using Tiles64 = mf64x4[NW <= 4 ? 5 : NW];

__device__ __forceinline__ double fast_rsqrt64(double x) {   // two Newton steps on the estimate
    double r = __builtin_amdgcn_rsq(x);
    r = r * fma(-0.5 * x * r, r, 1.5);
    return r * fma(-0.5 * x * r, r, 1.5);
}
__device__ __forceinline__ double uni(double x) { return lane_f64(x, 0); }

// Sums of two values (alike in the wave's lanes) over the waves.
template <int NW>
__device__ __forceinline__ cx<double> wg_sum64(LdsMfma64<NW>& L, int w, int& turn, double a, double b = 0.0) {
    if constexpr (NW == 1) return cx<double>{uni(a), uni(b)};
    turn ^= 1;
    if ((threadIdx.x & 63) == 0) {
        L.red[turn][w][0] = a;
        L.red[turn][w][1] = b;
    }
    __syncthreads();
    cx<double> s = {L.red[turn][0][0], L.red[turn][0][1]};
#pragma unroll
    for (int k = 1; k < NW; ++k) {
        s.re += L.red[turn][k][0];
        s.im += L.red[turn][k][1];
    }
    return cx<double>{uni(s.re), uni(s.im)};
}

// Complex sweep of all n pivots (diagonal stored minus 1; in the padding 0 on
// the diagonal, so an odd n's last pair is completed by the identity):
// (R, I) becomes -B^-1 + I.  neg: pivots that are not positive; pm: the
// smallest |determinant| of a pivot block.
template <int NW>
__device__ __forceinline__ void sweep_c64(LdsMfma64<NW>& L, Tiles64<NW>& R, Tiles64<NW>& I, int n, int w, int lane,
                                          int& neg, double& pm) {
    neg = 0;
    pm = 1.0e300;
    const int i = lane & 3, q = lane >> 4;
    // this lane's entry of the negated real form of the 2 x 2 inverse
    // [[i00, i01], [conj i01, i11]] acting on (re 0, re 1, im 0, im 1)
    const double al = i == q && (i & 1) == 0 ? -1.0 : 0.0, ga = i == q && (i & 1) == 1 ? -1.0 : 0.0;
    const double be = (i ^ q) == 1 ? -1.0 : 0.0;
    const double de = (i == 1 && q == 2) || (i == 2 && q == 1) ? -1.0
                      : (i == 0 && q == 3) || (i == 3 && q == 0) ? 1.0 : 0.0;
    const uint64_t flip = lane < 32 ? 0ull : 0x8000000000000000ull;
    int turn = 0;
    __syncthreads();   // the buffers' last use is over
    for (int K = 0; K < NW; ++K) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int s = 0; s < 4; s += 2) {
                if (16 * K + 4 * r + s < fresh(n)) {
                    double(*X)[64] = L.panel[turn];
                    turn ^= 1;
                    if (w == K && (q & 2) == s) {
                        const int at = lane & 31;   // quarter s, then s + 1
#pragma unroll
                        for (int J = 0; J < NW; ++J) {
                            X[J][at] = R[J][r];
                            X[J][32 + at] = I[J][r];
                        }
                    }
                    __syncthreads();
                    const double* D = &X[K][4 * r + s];
                    const double d00 = D[0] + 1.0, d01r = D[1], d01i = D[33], d11 = D[17] + 1.0;
                    const double det = fma(-d01r, d01r, fma(-d01i, d01i, d00 * d11));
                    const double rd = fast_rcp(det);
                    neg += (d00 > 0.0 ? 0 : 1) + (det * d00 > 0.0 ? 0 : 1);
                    pm = fmin(pm, fabs(det));
                    const double num = fma(al, d11, fma(ga, d00, fma(-be, d01r, -de * d01i)));
                    const double ca = num * rd;
                    const double v = __builtin_amdgcn_mfma_f64_4x4x4f64(ca, X[w][lane], 0.0, 0, 0, 0);
                    const double vm = __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ flip);
                    double b[NW], c[NW];
#pragma unroll
                    for (int J = 0; J < NW; ++J) {
                        b[J] = X[J][lane];
                        c[J] = X[J][lane ^ 32];
                    }
#pragma unroll
                    for (int J = 0; J < NW; ++J) {
                        R[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, b[J], R[J], 0, 0, 0);
                        I[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(vm, c[J], I[J], 0, 0, 0);
                    }
                }
            }
    }
    __syncthreads();
    neg = __builtin_amdgcn_readfirstlane(neg);
    pm = uni(pm);
}

// Real sweep of |Gamma| - shift by panels of four (see sweep64_wg): M becomes
// -A^-1 + I.  Returns whether every pivot was positive.
template <int NW>
__device__ __forceinline__ bool sweep_r64(LdsMfma64<NW>& L, Tiles64<NW>& M, int n, int w, int lane) {
    bool ok = true;
    const int i = lane & 3, q = lane >> 4;
    int turn = 0;
    __syncthreads();
    for (int K = 0; K < NW; ++K) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (16 * K + 4 * r < fresh(n) && ok) {
                double(*X)[64] = L.panel[turn];
                turn ^= 1;
                if (w == K) {
#pragma unroll
                    for (int J = 0; J < NW; ++J) X[J][lane] = M[J][r];
                }
                __syncthreads();
                const double* D = &X[K][4 * r];   // D[q][t] at 16 q + t
                const double a00 = D[0] + 1.0, a01 = D[1], a11 = D[17] + 1.0;
                const double b00 = D[2], b01 = D[3], b10 = D[18], b11 = D[19];
                const double c00 = D[34] + 1.0, c01 = D[35], c11 = D[51] + 1.0;
                const double da = fma(-a01, a01, a00 * a11), ra = fast_rcp(da);
                const double e00 = a11 * ra, e01 = -a01 * ra, e11 = a00 * ra;
                const double t00 = fma(e00, b00, e01 * b10), t01 = fma(e00, b01, e01 * b11);
                const double t10 = fma(e01, b00, e11 * b10), t11 = fma(e01, b01, e11 * b11);
                const double s00 = fma(-b00, t00, fma(-b10, t10, c00));
                const double s01 = fma(-b00, t01, fma(-b10, t11, c01));
                const double s11 = fma(-b01, t01, fma(-b11, t11, c11));
                const double ds = fma(-s01, s01, s00 * s11), rs = fast_rcp(ds);
                ok = __all((a00 > 0.0) & (da > 0.0) & (s00 > 0.0) & (ds > 0.0));
                const double f00 = s11 * rs, f01 = -s01 * rs, f11 = s00 * rs;
                const double g00 = fma(t00, f00, t01 * f01), g01 = fma(t00, f01, t01 * f11);
                const double g10 = fma(t10, f00, t11 * f01), g11 = fma(t10, f01, t11 * f11);
                const double h00 = fma(g00, t00, fma(g01, t01, e00));
                const double h01 = fma(g00, t10, fma(g01, t11, e01));
                const double h11 = fma(g10, t10, fma(g11, t11, e11));
                const bool i0 = (i & 1) == 0, q0 = (q & 1) == 0;
                const double tl = i0 ? (q0 ? h00 : h01) : (q0 ? h01 : h11);
                const double br = i0 ? (q0 ? f00 : f01) : (q0 ? f01 : f11);
                const double tr = i0 ? (q0 ? g00 : g01) : (q0 ? g10 : g11);
                const double bl = q0 ? (i0 ? g00 : g01) : (i0 ? g10 : g11);
                const double ca = i < 2 ? (q < 2 ? -tl : tr) : (q < 2 ? bl : -br);
                const double v = __builtin_amdgcn_mfma_f64_4x4x4f64(ca, X[w][lane], 0.0, 0, 0, 0);
                double b[NW];
#pragma unroll
                for (int J = 0; J < NW; ++J) b[J] = X[J][lane];
#pragma unroll
                for (int J = 0; J < NW; ++J) M[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, b[J], M[J], 0, 0, 0);
            }
        }
    }
    __syncthreads();
    return ok;
}

// Vectors: component lane + 64 t of x[t], held by every wave.
template <int NW> struct Eig64 {
    static constexpr int NC = (16 * NW + 63) / 64;
    cx<double> x[NC];
    double theta, dn, q;
    bool done;
};

// y = M x
template <int NW>
__device__ __forceinline__ void apply_64(LdsMfma64<NW>& L, const Tiles64<NW>& R, const Tiles64<NW>& I,
                                         const cx<double> (&x)[Eig64<NW>::NC], cx<double> (&y)[Eig64<NW>::NC], int w,
                                         int lane, int& turn) {
    constexpr int NC = Eig64<NW>::NC;
#pragma unroll
    for (int t = 0; t < NC; ++t)
        if (t == w / 4 && (lane >> 4) == (w & 3)) L.x[w][lane & 15] = x[t];
    wsync();
    const bool odd = lane & 1;
    double a1[4], a2[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {   // A: rows re x, im x against M, and im x, -re x against the imaginary part
        const cx<double> v = L.x[w][4 * r + (lane >> 4)];
        a1[r] = odd ? v.im : v.re;
        a2[r] = odd ? -v.re : v.im;
    }
    turn ^= 1;
    double* P = (double*)L.part[turn][w];
#pragma unroll
    for (int J = 0; J < NW; ++J) {
        double acc = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc = __builtin_amdgcn_mfma_f64_4x4x4f64(a1[r], R[J][r], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f64_4x4x4f64(a2[r], I[J][r], acc, 0, 0, 0);
        }
        if (lane < 32) P[2 * (16 * J + (lane & 15)) + (lane >> 4)] = acc;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NC; ++t) {
        const int c = lane + 64 * t;
        y[t] = cx<double>{0.0, 0.0};
        if (c < 16 * NW) {
            y[t] = L.part[turn][0][c];
#pragma unroll
            for (int k = 1; k < NW; ++k) y[t] = cadd(y[t], L.part[turn][k][c]);
        }
    }
}

template <int NW> __device__ __forceinline__ double norm2_64(const cx<double> (&x)[Eig64<NW>::NC]) {
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < Eig64<NW>::NC; ++t) s += cabs2(x[t]);
    return uni(sumR<64>(s));
}

// One normalised step (see step_wg); returns the squared change.
template <int NW>
__device__ __forceinline__ double step_64(Eig64<NW>& E, const cx<double> (&y)[Eig64<NW>::NC]) {
    constexpr int NC = Eig64<NW>::NC;
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < NC; ++t) s = fma(y[t].re, E.x[t].re, fma(y[t].im, E.x[t].im, s));
    E.theta = uni(sumR<64>(s));
    const double it = fast_rcp(E.theta);
    cx<double> d[NC];
#pragma unroll
    for (int t = 0; t < NC; ++t) d[t] = cx<double>{fma(y[t].re, it, -E.x[t].re), fma(y[t].im, it, -E.x[t].im)};
    const double d2 = norm2_64<NW>(d);
    const double k = fast_rsqrt64(1.0 + d2);
#pragma unroll
    for (int t = 0; t < NC; ++t) E.x[t] = cx<double>{(E.x[t].re + d[t].re) * k, (E.x[t].im + d[t].im) * k};
    return d2;
}

// Inverse iteration with B^-1 = I - M (see iterate_wg; the predicted error
// goes below 1e-11, or tol when polishing).
constexpr double kTol64 = 1.0e-11;
constexpr int kRounds64 = 36;
template <int NW>
__device__ __forceinline__ void iterate_64(LdsMfma64<NW>& L, const Tiles64<NW>& R, const Tiles64<NW>& I, int w, int lane,
                                           int& turn, double qb, int most, Eig64<NW>& E,
                                           double tol = kTol64) {
    constexpr int NC = Eig64<NW>::NC;
    double dp = 0.0;
    if (!(qb > 0.0)) E.q = 0.0;
    cx<double> y[NC];
    for (int k = qb > 0.0 ? 0 : -2; k < most; ++k) {
        apply_64<NW>(L, R, I, E.x, y, w, lane, turn);
#pragma unroll
        for (int t = 0; t < NC; ++t) y[t] = csub(E.x[t], y[t]);
        if (k < 0) {
            const double nr = k < -1 ? 1.0 : fast_rsqrt64(norm2_64<NW>(y));
#pragma unroll
            for (int t = 0; t < NC; ++t) E.x[t] = cscale(y[t], nr);
            continue;
        }
        const double d2 = step_64<NW>(E, y);
        const double dn = sqrt(d2);
        E.dn = dn;
        E.done = false;
        if (!(dn < 1.0e300)) return;   // not finite
        if (qb > 0.0) {
            E.done = dn * qb < tol * (1.0 - qb);
            if (E.done) return;
            continue;
        }
        if (dn < kTol64) E.done = true;
        if (k > 0) {
            E.q = dn / dp;
            const double q = fmin(E.q, 0.99);
            if (dn * q < kTol64 * (1.0 - q)) E.done = true;
            if (k > 1 && E.q > (double)kSlow && dn > 1.0e-5 && !E.done) return;
        }
        if (E.done) return;
        dp = dn;
    }
}

// Above 96 dates a wave's tiles leave few registers: loads of one tile at a
// time are in flight (all of them at once spilled).
template <int NW> __device__ __forceinline__ void tile_fence() {
    if constexpr (NW >= 7) __builtin_amdgcn_sched_barrier(0);
}

template <int NW>
__device__ __forceinline__ void load_gamma64(const GammaBuf64& gam, int n, int w, int lane, Tiles64<NW>& R,
                                             Tiles64<NW>& I) {
#pragma unroll
    for (int J = 0; J < NW; ++J) {
        int o = fresh_lane(gam.offset(16 * w + (lane >> 4), 16 * J + (lane & 15)));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const cx<double> g = gam.at(o);
            o += 4 * n * 16;
            R[J][r] = g.re;
            I[J][r] = g.im;
        }
        tile_fence<NW>();
    }
}

// |Gamma|, diagonal stored minus 1 and less shift (0 stored in the padding);
// false when an entry is not finite.
template <int NW>
__device__ __forceinline__ bool load_abs_64(LdsMfma64<NW>& L, const GammaBuf64& gam, int n, int w, int lane, double shift,
                                            int& turn, Tiles64<NW>& M) {
    double sum = 0.0;
#pragma unroll
    for (int J = 0; J < NW; ++J) {
        int o = fresh_lane(gam.offset(16 * w + (lane >> 4), 16 * J + (lane & 15)));
        const int dr = fresh_lane(16 * (J - w) + (lane & 15) - (lane >> 4));   // 4 r on the diagonal
        const double dv = 16 * J + (lane & 15) < n ? -shift : 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const cx<double> g = gam.at(o);
            o += 4 * n * 16;
            double v = sqrt(g.re * g.re + g.im * g.im);
            if (dr == 4 * r) v = dv;
            sum += v;
            M[J][r] = v;
        }
        tile_fence<NW>();
    }
    return wg_sum64<NW>(L, w, turn, __all(sum < 1.0e300) ? 0.0 : 1.0).re == 0.0;
}

// One pixel on the NW waves of a workgroup.
// keep: LDS for the wave's share of the inverse of |Gamma| (kKeep64<NW>: each
// lane's own entries, 8 N^2 bytes for the workgroup); above 80 dates that
// would leave one workgroup per CU, and the sweep, a quarter of the complex
// one's work, is run again for each shift instead.
template <int NW> constexpr bool kKeep64 = NW <= 5;

template <int MODE, int NW>
__device__ __forceinline__ void solve_mfma64_pixel(const SolveArgs& a, LdsMfma64<NW>& L, double* keep, int w, int lane_in,
                                                   int np, const GammaBuf64& gam, long long pix) {
    constexpr int NC = Eig64<NW>::NC;
    const int n = gam.n;
    const bool stbas = a.method == FRINGE_METHOD_STBAS && MODE == MODE_EVD;
    int code = 0;
    bool inv = MODE != MODE_EVD;
    int turn = 0;
    Eig64<NW> E;
    const bool act = np >= 0;
    // What follows from the lane is computed again in each stage: held over
    // the sweeps it spilled.
    if (act) {
        const int lane = fresh_lane(lane_in), c16 = lane & 15, q = lane >> 4;
        if constexpr (MODE == MODE_MLE) {
            Tiles64<NW> R, I;
            load_gamma64<NW>(gam, n, w, lane, R, I);
            double sum = 0.0;
            const int rd = (c16 - q) & 3 ? -1 : (c16 - q) >> 2;   // register of the diagonal in tile (w, w)
            const bool own = 16 * w + c16 < n;
#pragma unroll
            for (int J = 0; J < NW; ++J)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sum += fabs(R[J][r]) + fabs(I[J][r]);
                    if (J == w && r == rd) R[J][r] = own ? -1.0e-6 : 0.0;   // 1 - 1e-6, stored minus 1
                }
            if (wg_sum64<NW>(L, w, turn, __all(sum < 1.0e300) ? 0.0 : 1.0).re != 0.0) {
                code = -1;
            } else {
                int neg;
                double pm;
                sweep_c64<NW>(L, R, I, n, w, lane, neg, pm);
                if (neg) code = -2;   // an eigenvalue of Gamma below 1e-6
            }
            if (code == 0) {
                Tiles64<NW> M;
                load_abs_64<NW>(L, gam, n, w, lane, 1.0e-6, turn, M);
                if (!sweep_r64<NW>(L, M, n, w, lane)) code = -4;
            }
        }
        if constexpr (MODE != MODE_EVD) {
            if (code == 0) {
                Tiles64<NW> M;   // -|Gamma|^-1 + I
                if (!load_abs_64<NW>(L, gam, n, w, lane, 0.0, turn, M)) {
                    code = -1;
                } else {
                    const bool pd = sweep_r64<NW>(L, M, n, w, lane);
                    if (MODE == MODE_EMI) inv = pd;   // else the EVD fallback
                    else if (!pd) code = -5;
                    if constexpr (kKeep64<NW>)
#pragma unroll
                        for (int J = 0; J < NW; ++J)
#pragma unroll
                            for (int r = 0; r < 4; ++r) keep[(4 * NW * w + 4 * J + r) * 64 + lane] = M[J][r];
                }
            }
        }
    }

    // ---- the eigenpair ----
    if (act && code == 0) {
        double sigma = 1.0, sg = 1.0;
        // H is positive semidefinite, so its eigenvalues lie past 0; `good` is a
        // shift that no eigenvalue lies before, `up` one that some lie before
        double good = 0.0, up = 1.0e300;
        auto fresh_start = [&](int kind) {
            const int lane = fresh_lane(lane_in);
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const int c = lane + 64 * t;
                // the phases of the middle column, or arbitrary ones
                const cx<double> g = gam.at(gam.offset(n >> 1, c));
                const uint32_t u = (uint32_t)(c + 1) * 2654435761u + (uint32_t)kind * 40503u;
                const double re = kind == 0 ? g.re : (double)(u >> 20) - 2048.0;
                const double im = kind == 0 ? -g.im : (double)((u >> 8) & 4095u) - 2047.5;
                const double g2 = re * re + im * im;
                const bool z = !(g2 > 1.0e-290);
                const double s = fast_rsqrt64(z ? 1.0 : g2);
                E.x[t].re = c < n ? (z ? 1.0 : re * s) : 0.0;
                E.x[t].im = c < n && !z ? im * s : 0.0;
            }
            const double nr = fast_rsqrt64(norm2_64<NW>(E.x));
#pragma unroll
            for (int t = 0; t < NC; ++t) E.x[t] = cscale(E.x[t], nr);
        };
        fresh_start(0);
        if (!inv) {
            const int lane = fresh_lane(lane_in), c16 = lane & 15, q = lane >> 4;
            sg = -1.0;
            Tiles64<NW> R, I;
            load_gamma64<NW>(gam, n, w, lane, R, I);
            double f2 = 0.0;
            const int d0 = c16 - q - 16 * w;
#pragma unroll
            for (int J = 0; J < NW; ++J)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (stbas && abs(4 * r - d0 - 16 * J) > a.bw) {
                        R[J][r] = 0.0;
                        I[J][r] = 0.0;
                    }
                    f2 = fma(R[J][r], R[J][r], fma(I[J][r], I[J][r], f2));
                }
            f2 = wg_sum64<NW>(L, w, turn, uni(sumR<64>(f2))).re;
            if (!(f2 < 1.0e300)) code = -6;
            // no eigenvalue lies above the mean, 1, plus sqrt(n - 1) deviations
            // (1e-14: what rounding can take from the squared deviation)
            good = 1.0 + sqrt((fmax(f2 * (1.0 / n) - 1.0, 0.0) + lit(1.0e-14)) * (double)(n - 1)) + 1.0e-9;
            up = -1.0e300;
            if (code == 0) {
                cx<double> y[NC];
                double d2 = 1.0;
                for (int k = 0; k < 4; ++k) {
                    apply_64<NW>(L, R, I, E.x, y, w, lane, turn);
                    d2 = step_64<NW>(E, y);
                }
                sigma = fmin(E.theta + fabs(E.theta) * fmax(sqrt(d2), 0.02), good);
            }
        }
        double lam = 0.0;
        // Each round sweeps at one shift; the bracket (good, up] halves at
        // least wherever the suggested shift leaves it, so the rounds isolate
        // the extreme eigenvalue, unless it is nearly a multiple one.  The last
        // rounds then take the bracket's end that no eigenvalue lies before (a
        // little further out each), and the vector of the eigenspace that
        // iteration from there finds.
        bool found = false;
        for (int att = 0; att < 40 && code == 0; ++att) {
            const bool late = att >= kRounds64;
            if (late) sigma = good - sg * lit(1.0e-9) * (1.0 + fabs(good)) * (double)(1 << 6 * (att - kRounds64));
            // ---- B = +-(A - sigma I), diagonal stored minus 1 ----
            Tiles64<NW> R, I;
            const int lane = fresh_lane(lane_in), c16 = lane & 15, q = lane >> 4;
            const int d0 = c16 - q - 16 * w, rdl = (c16 - q) & 3 ? -1 : (c16 - q) >> 2;
            const bool own = 16 * w + c16 < n;
            if (inv) {
                if constexpr (MODE != MODE_EVD) {
                    Tiles64<NW> M;
                    if constexpr (!kKeep64<NW>) {
                        load_abs_64<NW>(L, gam, n, w, lane, 0.0, turn, M);
                        sweep_r64<NW>(L, M, n, w, lane);
                    }
                    load_gamma64<NW>(gam, n, w, lane, R, I);
#pragma unroll
                    for (int J = 0; J < NW; ++J)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            double m;
                            if constexpr (kKeep64<NW>) m = -keep[(4 * NW * w + 4 * J + r) * 64 + lane];
                            else m = -M[J][r];
                            R[J][r] *= m;
                            I[J][r] *= m;
                            if (J == w && r == rdl) R[J][r] = own ? m - sigma : 0.0;
                        }
                }
            } else {
                load_gamma64<NW>(gam, n, w, lane, R, I);
#pragma unroll
                for (int J = 0; J < NW; ++J)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const double m = stbas && abs(4 * r - d0 - 16 * J) > a.bw ? 0.0 : -1.0;
                        R[J][r] *= m;
                        I[J][r] *= m;
                        if (J == w && r == rdl) R[J][r] = own ? sigma - 2.0 : 0.0;
                    }
            }
            int neg;
            double pm;
            sweep_c64<NW>(L, R, I, n, w, lane, neg, pm);
            double next;   // the next shift, from the two eigenvalues next to this one
            if (late) {
                if (neg != 0) continue;
            } else if (neg == 0) {
                good = sg * (sigma - good) > 0.0 ? sigma : good;
            } else {
                up = sg * (sigma - up) < 0.0 ? sigma : up;
            }
            if (neg > 1) {
                next = 0.5 * (good + sigma);
            } else {
                iterate_64<NW>(L, R, I, w, lane, turn, 0.0, att < 8 ? 24 : 60, E);
                const double mu = 1.0 / E.theta;
                lam = sigma + sg * mu;
                if (!(fabs(lam) < 1.0e300) || !(E.dn < 1.0e300) || pm < 1.0e-14) {   // the shift is an eigenvalue
                    sigma -= sg * lit(1.0e-7) * (1.0 + fabs(sigma)) * (double)(1 << min(2 * att, 24));
                    bool bad = false;
#pragma unroll
                    for (int t = 0; t < NC; ++t) bad = bad || !(cabs2(E.x[t]) < 1.0e300);
                    if (__any(bad)) fresh_start(0);
                    continue;
                }
                found = late;
                if (found) break;
                if (neg == 0 ? E.theta < 0.0 : E.theta > 0.0) {   // not the extreme one: it lies before the shift
                    fresh_start(att + 1);
                    next = 0.5 * (good + sigma);
                } else if (!E.done) {   // as in solve_mfma_pixel
                    const double qq = E.q > 0.0 ? fmin(fmax(E.q, 1.0e-3), 0.98) : 0.98;
                    const double gap = fabs(mu) / qq - mu;
                    const double e = fmin(E.dn * qq / (1.0 - qq), 1.0);
                    next = sigma + sg * (mu - (e * e + lit(0.15)) * gap);
                } else {
                    // the other eigenvalues of the inverse have squares that
                    // sum to s2: the vector's is the largest, and how fast it
                    // converges, follow
                    double f = 0.0;
#pragma unroll
                    for (int J = 0; J < NW; ++J)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const double x = J == w && r == rdl ? (own ? 1.0 - R[J][r] : 0.0) : R[J][r];
                            f = fma(x, x, fma(I[J][r], I[J][r], f));
                        }
                    f = wg_sum64<NW>(L, w, turn, uni(sumR<64>(f))).re;
                    const double qb = sqrt(fmax(f - E.theta * E.theta, 0.0)) * fabs(mu);
                    found = qb < lit(0.8);
                    if (found) {
                        // no phase off by more than 1e-8 rad: a component
                        // below 1e-3 takes more than kTol64
                        double m2 = 1.0;
#pragma unroll
                        for (int t = 0; t < NC; ++t)
                            if (lane + 64 * t < n) m2 = fmin(m2, cabs2(E.x[t]));
                        m2 = uni(minR<64>(m2));
                        const double tol = fmin(kTol64, fmax(lit(1.0e-8) * sqrt(m2), lit(2.0e-15)));
                        if (E.dn * qb > tol * (1.0 - qb)) iterate_64<NW>(L, R, I, w, lane, turn, qb, 60, E, tol);
                        break;
                    }
                    next = lam - sg * lit(0.1) * fabs(mu);   // closer, and before it
                }
            }
            next = uni(next);
            const double in0 = sg * (next - good), in1 = sg * (up - next);
            sigma = in0 > 0.0 && in1 > 0.0 ? next : fabs(up) < 1.0e299 ? 0.5 * (good + up) : good;
        }
        if (code == 0 && !found) code = MODE == MODE_EMI ? -1 : -6;   // (nothing but a matrix that is not finite)
        if (MODE != MODE_EMI && code == 0 && !(lam >= 1.0e-6)) code = -7;
    }

    const bool ok = act && code == 0;
    const int lane = fresh_lane(lane_in), c16 = lane & 15, q = lane >> 4;
    if (!ok) {
        if (w == 0) {
            for (int d = lane; d < n; d += 64) a.phase[(long long)d * a.npx + pix] = make_float2(0.0f, 0.0f);
            if (lane == 0) {
                a.tcorr[pix] = act ? (float)code : 0.0f;
                a.comp[pix] = make_float2(0.0f, 0.0f);
            }
        }
        return;
    }

    // ---- referenced phases (evd.cpp:738-749): every wave all dates ----
    cx<double> vref = {0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NC; ++t)
        if (t == a.ref / 64) vref = cx<double>{lane_f64(E.x[t].re, a.ref & 63), lane_f64(E.x[t].im, a.ref & 63)};
    bool okr, oku, okv;
    const cx<double> cref = unit_or(cconj(vref), cx<double>{1.0, 0.0}, okr);
    cx<double> cs = {0.0, 0.0};
    cx<float>* O = (cx<float>*)L.part[0];
    __syncthreads();   // part's last use is over
#pragma unroll
    for (int t = 0; t < NC; ++t) {
        const int c = lane + 64 * t;
        const cx<double> u = unit_or(cmulc(E.x[t], vref), cx<double>{0.0, 0.0}, oku);
        cx<double> o = oku ? u : (okr ? cref : unit_or(E.x[t], cx<double>{1.0, 0.0}, okv));
        if (c == a.ref) o = cx<double>{1.0, 0.0};
        const cx<float> of = {(float)o.re, (float)o.im};
        if (w == 0) {
            if (c < n) a.phase[(long long)c * a.npx + pix] = make_float2(of.re, of.im);
            if (c < 16 * NW) O[c] = of;
            // ---- compressed SLC (evd.cpp:755-762) ----
            if (c >= a.ref && c < n) {
                const float2 z = a.slc[(long long)c * a.npx + pix];
                cs.re += (double)(z.x * of.re + z.y * of.im);
                cs.im += (double)(z.y * of.re - z.x * of.im);
            }
        }
    }
    __syncthreads();
    // ---- temporal coherence (evd.cpp:770-786): the wave's rows against the
    // columns right of them, pairs j <= i + bw for STBAS ----
    double sr = 0.0, si = 0.0;
    for (int J = w; J < NW; ++J) {
        const int c = 16 * J + c16;
        const cx<float> oc = O[c];
        int off = gam.offset(16 * w + q, c);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * w + 4 * r + q;
            const cx<double> g = gam.at(off);
            off += 4 * n * 16;
            const cx<float> orow = O[row];
            const bool use = row < c && c < n && !(stbas && c - row > a.bw);
            const double g2 = cabs2(g);
            const bool z = !(g2 > 1.0e-290);   // a zero has phase 0
            const double rs = z ? 0.0 : fast_rsqrt64(g2);
            const cx<double> ph = z ? cx<double>{1.0, 0.0} : cx<double>{g.re * rs, g.im * rs};
            const cx<double> t = cmul(cmulc(ph, cx<double>{orow.re, orow.im}), cx<double>{oc.re, oc.im});
            if (use) {
                sr += t.re;
                si += t.im;
            }
        }
    }
    const cx<double> tc = wg_sum64<NW>(L, w, turn, uni(sumR<64>(sr)), uni(sumR<64>(si)));
    if (w == 0) {
        cs = cx<double>{sumR<64>(cs.re), sumR<64>(cs.im)};
        if (lane == 0) {
            a.tcorr[pix] = (float)(sqrt(tc.re * tc.re + tc.im * tc.im) * a.inv_pairs);
            a.comp[pix] = make_float2((float)(cs.re * a.inv_comp), (float)(cs.im * a.inv_comp));
        }
    }
}

// Waves per SIMD, as many as leave no register spilled (as in solve_mfma_wg.hpp).
constexpr int waves64(int nw) { return nw <= 1 ? 4 : nw <= 3 ? 3 : 2; }
// Dynamic LDS of the plain kernel.
template <int MODE, int NW> constexpr size_t keep64_bytes() {
    return MODE != MODE_EVD && kKeep64<NW> ? (size_t)NW * NW * 4 * 64 * sizeof(double) : 0;
}

template <int MODE, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(waves64(NW)))) void solve_mfma64_kernel(SolveArgs a) {
    __shared__ LdsMfma64<NW> L;
    extern __shared__ __align__(16) char smem[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int slot = a.slots - 1 - (int)blockIdx.x;   // last-first, as the other solvers
    const cx<double>* gam = (const cx<double>*)a.gamma + (size_t)slot * a.n * a.n;
    solve_mfma64_pixel<MODE, NW>(a, L, (double*)smem, w, lane, a.npix[slot], GammaBuf64(gam, a.n), a.first + slot);
}

// The re-solve: each workgroup loops over its share of the list, computes the
// pixel's FP64 coherence with the plain path's Gram into its global area and
// runs the chain on it.
template <int MODE, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(waves64(NW)))) void resolve_mfma64_kernel(SolveArgs a) {
    __shared__ union {
        LdsMfma64<NW> chain;
        LdsGram64<NW> gram;
    } L;
    extern __shared__ __align__(16) char smem[];
    const int w0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    cx<double>* gam = (cx<double>*)((char*)a.awork + a.awork_stride * (size_t)blockIdx.x);
    const int cnt = min(*a.list_count, a.list_cap);
    for (int e = blockIdx.x; e < cnt; e += gridDim.x) {
        const long long pix = a.list[e];
        // nothing derived from the lane or the divisors is worth registers across the loop
        const int lane = fresh_lane(threadIdx.x & 63), w = fresh(w0), n = fresh(a.n);
        GramArgs g = a.g64;
        g.cols = fresh(g.cols);
        g.Nx = fresh(g.Nx);
        const int np = gram_mfma64_pixel<NW>(g, L.gram, (int*)smem, w, lane, pix, gam);
        __threadfence();
        __syncthreads();
        solve_mfma64_pixel<MODE, NW>(a, L.chain, (double*)smem, w, lane, np, GammaBuf64(gam, n), pix);
        __syncthreads();
    }
}

// The plain path's coherence: one slot per workgroup.
template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW <= 4 ? 4 : NW <= 7 ? 3 : 2))) void gram_mfma64_kernel(GramArgs a) {
    __shared__ LdsGram64<NW> L;
    extern __shared__ __align__(16) char smem[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int slot = blockIdx.x;
    cx<double>* gam = (cx<double>*)a.gamma + (size_t)slot * a.n * a.n;
    const int np = gram_mfma64_pixel<NW>(a, L, (int*)smem, w, lane, a.first + slot, gam);
    if (threadIdx.x == 0) a.npix[slot] = np;
}

}  // namespace fringe
