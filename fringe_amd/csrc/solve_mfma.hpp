// solve_mfma.hpp -- FP32 estimator chain of the mixed precisions on the
// matrix cores, up to 32 dates, one pixel per wave.
//
// Every matrix of the pixel lives in the accumulator layout of
// v_mfma_f32_32x32x2 (lane l, register v: column l % 32, row
// 8 (v / 4) + 4 (l / 32) + v % 4) or, for the FP64 |Gamma|, of
// v_mfma_f64_16x16x4 (four 16 x 16 tiles; lane l, register r: column l % 16,
// row 4 r + l / 16).  In both a row of the matrix lies in the lanes of one
// register exactly as the instruction's B operand wants it, and a Hermitian
// matrix' column is the conjugate of that row, so an elimination step needs
// no data movement but a half swap.
//
// Inverses come from the symmetric sweep operator: for pivot row P (with
// P_k = A_kk - 1) every entry becomes A_rc - conj(P_r) P_c / A_kk, one rank-1
// update of the whole matrix on the matrix cores (complex FP32: two 32x32x2
// MFMAs a pivot, k = the real and imaginary parts; real FP64: four 16x16x4
// a pivot pair).  It leaves -A^-1 + 2 I; the diagonals are stored with 1
// subtracted throughout, which gives the P_k of the unswept rows for free.
//
// The wanted eigenpair of A (smallest of H = |Gamma|^-1 o Gamma, largest of
// Gamma) comes from inverse iteration with the explicit inverse of
// B = +-(A - sigma I): H has its smallest eigenvalue just above 1 when the
// phases close (the rows of A^-1 o A sum to 1), so sigma = 1 converges in a
// handful of 4 n^2-flop products; Gamma takes sigma just above its Rayleigh
// quotient after three power steps.  Slow convergence moves sigma.  Every
// pivot's sign is counted, and the inertia, the Frobenius norm of the
// inverse and the Rayleigh quotient certify that no other eigenvalue lies
// within the certification distance (cert_eps).
//
// What bounds it: the vector unit and the FP32 / FP64 matrix instructions
// together (65 and 42 % of the kernel's cycles at 30 dates; 4, 5 or 6 waves
// per SIMD measured the same).  There a pixel takes 2.55 k vector
// instructions and 135 MFMAs, against 9.2 k vector instructions in the
// tridiagonalising two-pixel solver it replaced.  Solve stage of a 2048 x
// 2048 tile at 30 dates (EMI): 67.5 ms before, 31.2 ms now (29.5 before
// refine32); of a 640 x 640 tile at 20 dates (MLE): 7.4 ms before, 3.1 ms now.
//
// Up to 16 dates the same chain runs on one 16 x 16 tile (four registers a
// matrix instead of sixteen, 16x16x4 MFMAs that take two pivots each): 256 x
// 256 pixels of 10 dates (EVD) 0.21 -> 0.16 ms, 64 x 64 of 8 0.020 -> 0.017.
#pragma once
#include "link_solve.hpp"
#include "solve32.hpp"

namespace fringe {

typedef float mf32x16 __attribute__((ext_vector_type(16)));
typedef double mf64x4 __attribute__((ext_vector_type(4)));

// Certification distance: no eigenvalue may lie within scale eps |A| / min_t
// |v_t| of the selected one, |A| bounded by the eigenvalues' mean and
// deviation (1.2-1.6 times the norm).  A certified phase is then wrong by C /
// scale at most, where C, the error times gap min|v| / (eps |A|), was measured
// against the FP64 path on stacks of 5 to 128 dates and 12 to 130 looks, with
// coherences that decay to 0, to 0.2, 0.9 and 0.99, noise alone, and two
// scatterers.
//
// Gamma: C is 1.8 at 5 dates, 1.25 at 8, 1.13 at 12, 0.8 at 16 and 20, 0.54 at
// 30, 0.41 at 40, 0.3 at 64 and 0.22 at 96 and more (the tridiagonalising FP32
// solver's, at 1e4: 2.4 to 6.0).  So kCertScale up to 8 dates falls as 1 / n to
// kCertScaleG at 32: errors of 2.1e-4 rad at most, and less than that solver's
// at every n.  kCertScale throughout, with the bound on |A|, left more pixels
// to FP64 than that solver did (48 k pixels of 128 dates, EVD: 14.8 k, that
// solver 9.1 k, now 3.1 k; solver and re-solve 40.0 -> 22.3 ms).
//
// H below |H| = 100: C is 1.0 up to 8 dates, 0.5 up to 12, 0.3 up to 20, 0.17
// at 30, 0.08 at 48 and 0.03 at 96, a third to a seventh of that solver's, so a
// scale of 3e3, falling as 1 / n from 48 dates on, keeps to its worst error
// (3.7e-4 rad at 8 dates, 8e-5 at 30, 2e-5 from 48 on).  C grows with the root
// of |H| beyond (Gamma's own error, multiplied by the inverse of |Gamma|: 0.5
// at 16 dates and |H| = 1000), and so does the scale, up to kCertScale.
// Against kCertScale for H everywhere: 46.6 k pixels of 48 dates 8.0 -> 3.9
// ms, 65.5 k of 96 78 -> 54 (51 with Gamma's).
//
// Both hold for Gamma from half pairs (22 bits): bfloat16 pairs carry 16, and
// take kCertScale throughout.
constexpr float kCertScaleH = 3.0e3f, kCertScaleG = 2.5e3f;
__device__ __forceinline__ float cert_eps(bool inv, float cert_h, float cert_g, float tn) {
    const float most = kCertScale * Lim<float>::eps();
    return inv ? fminf(cert_h * __builtin_amdgcn_sqrtf(fmaxf(0.01f * tn, 1.0f)), most) : cert_g;
}

// Accumulator of a DIM x DIM matrix: NV registers, lane l holds column l % DIM
// and, with h = l / DIM, rows row(v, h).
template <int DIM> struct Acc;
template <> struct Acc<32> {
    typedef mf32x16 type;
    static constexpr int NV = 16;
    static __device__ __forceinline__ constexpr int row(int v, int h) { return 8 * (v / 4) + 4 * h + v % 4; }
};
template <> struct Acc<16> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int NV = 4;
    static __device__ __forceinline__ constexpr int row(int v, int h) { return 4 * h + v; }
};

template <int DIM> struct LdsMfma {
    static constexpr int S = DIM + 4;   // row stride of T: 16-byte rows of four, spread over the banks
    float T[DIM * S];   // |Gamma|^-1, row-major
    float xr[DIM], xi[DIM];
};

__device__ __forceinline__ float lane_f32(float x, int lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), lane));
}
__device__ __forceinline__ double lane_f64(double x, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// (a.lo | b.lo) and (a.hi | b.hi), halves of 32 lanes
__device__ __forceinline__ void swap32(float a, float b, float& lo, float& hi) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    lo = __uint_as_float(s[0]);
    hi = __uint_as_float(s[1]);
}
__device__ __forceinline__ float both32(float x) {   // x.lo + x.hi in both halves
    float lo, hi;
    swap32(x, x, lo, hi);
    return lo + hi;
}
// a scalar the compiler has to look at afresh: comparisons with it stay where
// they are instead of being hoisted into (spilled) scalar registers
__device__ __forceinline__ int fresh(int x) {
    asm volatile("" : "+s"(x));
    return x;
}
__device__ __forceinline__ int fresh_lane(int x) {   // the same for a lane value
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ int lane_now() {   // the lane's number, held in no register until here
    int x;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
    return x;
}
__device__ __forceinline__ float scal(float x) {   // a value alike in all lanes, in a scalar register
    asm volatile("" : "+v"(x));   // (else the arithmetic is moved behind the read and stays in a vector register)
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}
template <typename T> __device__ __forceinline__ T lit(T x) {   // a constant, likewise
    asm volatile("" : "+s"(x));
    return x;
}
// a uniform value as a scalar (control flow and scalar operands)
__device__ __forceinline__ float uni(float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); }

// Complex sweep of all n pivots (diagonal stored minus 1, rows and columns
// from n on zero): (R, I) becomes -B^-1 + I.  neg: pivots that are not
// positive; near: the smallest distance of a stored pivot p - 1 from -1, in
// units of the last place (p >= 1e-4 when it is at least 1700).  Both are
// kept in scalar integer arithmetic, off the vector unit.
__device__ __forceinline__ void sweep32(mf32x16& R, mf32x16& I, int n, int lane, int& neg, int& near) {
    neg = 0;
    near = 0x7fffffff;
    const uint32_t flip = lane < 32 ? 0u : 0x80000000u;
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int j = 8 * (v / 4) + 4 * h + v % 4;
            if (j < fresh(n)) {
                const int pb = __builtin_amdgcn_readlane(__float_as_int(R[v]), j + 32 * h);
                neg += (uint32_t)pb < 0xBF800000u ? 0 : 1;   // p - 1 > -1
                near = min(near, abs(pb - (int)0xBF800000));
                const float q = -__builtin_amdgcn_rcpf(__int_as_float(pb) + 1.0f);
                float b[2], c[2];
                swap32(R[v], I[v], b[0], b[1]);   // (re | im) of the pivot row
                swap32(I[v], R[v], c[0], c[1]);   // (im | re)
                const float a = b[h] * q;         // (re | im) of -conj(P) / p for the real part,
                const float d = __uint_as_float(__float_as_uint(a) ^ flip);   // (re | -im) for the imaginary one
                R = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b[h], R, 0, 0, 0);
                I = __builtin_amdgcn_mfma_f32_32x32x2f32(d, c[h], I, 0, 0, 0);
            }
        }
}

// The same for a matrix of 16 x 16, by pairs of pivots 8 rows apart: a swap of
// 16-lane rows puts (re | im) of the two pivot rows into the four k of one
// 16x16x4 MFMA.  With D the pivots' 2 x 2 block, W = D^-1 times the rows is a
// combination of the lane's own word, the other row's and the other row's
// other part.
__device__ __forceinline__ void sweep32(Acc<16>::type& R, Acc<16>::type& I, int n, int lane, int& neg, int& near) {
    neg = 0;
    near = 0x7fffffff;
    const uint32_t odd = (lane & 16) << 27;                          // the imaginary parts' lanes
    const uint32_t gam = lane < 16 || lane >= 48 ? 0x80000000u : 0u;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int p0 = v + 4 * s, p1 = p0 + 8;
            if (p0 < fresh(n)) {
                const float r = R[v], i = I[v];
                const float d00 = lane_f32(r, 16 * s + p0) + 1.0f, d11 = lane_f32(r, 16 * (s + 2) + p1) + 1.0f;
                const float x = lane_f32(r, 16 * s + p1), y = lane_f32(i, 16 * s + p1);
                const float det = fmaf(-x, x, fmaf(-y, y, d00 * d11));
                const float rd = __builtin_amdgcn_rcpf(det);
                const int pa = __builtin_amdgcn_readfirstlane(__float_as_int(d00 - 1.0f));
                const int pb = __builtin_amdgcn_readfirstlane(__float_as_int(fmaf(det, __builtin_amdgcn_rcpf(d00), -1.0f)));
                neg += ((uint32_t)pa < 0xBF800000u ? 0 : 1) + ((uint32_t)pb < 0xBF800000u ? 0 : 1);
                near = min(near, min(abs(pa - (int)0xBF800000), abs(pb - (int)0xBF800000)));
                const auto bb = __builtin_amdgcn_permlane16_swap(__float_as_uint(r), __float_as_uint(i), false, false);
                const auto cc = __builtin_amdgcn_permlane16_swap(__float_as_uint(i), __float_as_uint(r), false, false);
                const float b = __uint_as_float(bb[s]), c = __uint_as_float(cc[s]);
                float lo, hi;
                swap32(b, b, lo, hi);
                const float bo = lane < 32 ? hi : lo;   // the other pivot's row
                swap32(c, c, lo, hi);
                const float co = lane < 32 ? hi : lo;   // its other part
                const float al = (lane < 32 ? d11 : d00) * -rd;
                const float ga = __uint_as_float(__float_as_uint(y * rd) ^ gam);
                const float a = fmaf(al, b, fmaf(x * rd, bo, ga * co));
                const float d = __uint_as_float(__float_as_uint(a) ^ odd);
                R = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, R, 0, 0, 0);
                I = __builtin_amdgcn_mfma_f32_16x16x4f32(d, c, I, 0, 0, 0);
            }
        }
}

// Over a column's lanes, result in all of them; over the row groups of lanes.
template <int DIM, typename Op, typename T> __device__ __forceinline__ T redC(T x) {
    if constexpr (DIM == 32) return red32<Op>(x);
    else return red16<Op>(x);
}
template <int DIM> __device__ __forceinline__ float sumH(float x) {
    if constexpr (DIM == 16) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        x = __uint_as_float(s[0]) + __uint_as_float(s[1]);
    }
    return both32(x);
}

// x of the rows a lane's registers hold, from LDS
template <int DIM>
__device__ __forceinline__ void row_values(const LdsMfma<DIM>& L, int h, float (&xr)[Acc<DIM>::NV],
                                           float (&xi)[Acc<DIM>::NV]) {
#pragma unroll
    for (int a = 0; a < Acc<DIM>::NV / 4; ++a) {
        const float4 p = *(const float4*)&L.xr[8 * a + 4 * h];
        const float4 q = *(const float4*)&L.xi[8 * a + 4 * h];
        xr[4 * a] = p.x; xr[4 * a + 1] = p.y; xr[4 * a + 2] = p.z; xr[4 * a + 3] = p.w;
        xi[4 * a] = q.x; xi[4 * a + 1] = q.y; xi[4 * a + 2] = q.z; xi[4 * a + 3] = q.w;
    }
}

// y = M x for Hermitian (R, I): component c of x and y in lanes c, c + DIM, ...
template <int DIM>
__device__ __forceinline__ cx<float> apply32(LdsMfma<DIM>& L, const typename Acc<DIM>::type& R,
                                             const typename Acc<DIM>::type& I, cx<float> x, int col, int h) {
    constexpr int NV = Acc<DIM>::NV;
    if (h == 0) {
        L.xr[col] = x.re;
        L.xi[col] = x.im;
    }
    wsync();
    float xr[NV], xi[NV];
    row_values<DIM>(L, h, xr, xi);
    float re[2] = {0.0f, 0.0f}, im[2] = {0.0f, 0.0f};
#pragma unroll
    for (int v = 0; v < NV; ++v) {   // conj(M_rc) x_r
        re[v & 1] = fmaf(R[v], xr[v], re[v & 1]);
        im[v & 1] = fmaf(R[v], xi[v], im[v & 1]);
        re[v & 1] = fmaf(I[v], xi[v], re[v & 1]);
        im[v & 1] = fmaf(-I[v], xr[v], im[v & 1]);
    }
    wsync();
    return cx<float>{sumH<DIM>(re[0] + re[1]), sumH<DIM>(im[0] + im[1])};
}

// One pixel's n x n coherence through a buffer descriptor: its bounds check
// reads rows >= n as zero, and lanes of columns >= n are given an offset
// outside it, so no load needs a comparison.
struct GammaBuf {
    __amdgpu_buffer_rsrc_t rsrc;
    int n;
    __device__ __forceinline__ GammaBuf(const cx<float>* gam, int n_) : n(n_) {
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)gam, 0, n_ * n_ * 8, 0x00027000);
    }
    __device__ __forceinline__ int offset(int row, int c) const { return c < n ? (row * n + c) * 8 : 0x40000000; }
    __device__ __forceinline__ cx<float> at(int off) const {
        const auto u = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
        return cx<float>{__uint_as_float(u[0]), __uint_as_float(u[1])};
    }
};

// Gamma in the accumulator layout; rows and columns >= n read as zero
template <int DIM>
__device__ __forceinline__ void load_gamma32(const GammaBuf& gam, int n, int col, int h, typename Acc<DIM>::type& R,
                                             typename Acc<DIM>::type& I) {
    int o = fresh_lane(gam.offset(4 * h, col));   // (offsets are not worth registers from one load to the next)
#pragma unroll
    for (int v = 0; v < Acc<DIM>::NV; ++v) {
        const cx<float> g = gam.at(o);
        o += (v % 4 == 3 ? 5 : 1) * n * 8;
        R[v] = g.re;
        I[v] = g.im;
    }
}

struct EigState {
    cx<float> x;     // unit vector, component col
    float theta;     // Rayleigh quotient of B^-1
    float dn, q;     // last step's change and contraction
    float dq;        // the change that q was measured with
    bool done;
};

// Inverse iteration with B^-1 = I - M: two plain products (the start vector
// is far off), then normalised steps until the error predicted behind one more
// (refine32's) is below 4e-7, or until the contraction proves worse than kSlow
// (moving the shift then costs less than going on).
constexpr float kSlow = 0.35f;
constexpr int kNearInside = 1600000;   // |pivot| >= 0.1
// qb > 0: polishing instead, until the error predicted from the contraction
// qb that the spectrum allows is below 4e-7.
template <int DIM>
__device__ __forceinline__ void iterate32(LdsMfma<DIM>& L, const typename Acc<DIM>::type& R,
                                          const typename Acc<DIM>::type& I, int col, int h, float qb, EigState& E) {
    float dp = 0.0f;
    if (!(qb > 0.0f)) E.q = E.dq = 0.0f;
    for (int k = qb > 0.0f ? 0 : -2; k < 24; ++k) {
        const cx<float> y = csub(E.x, apply32<DIM>(L, R, I, E.x, col, h));
        if (k < 0) {
            const float nr = k < -1 ? 1.0f : __builtin_amdgcn_rsqf(uni(redC<DIM, OpAdd>(cabs2(y))));
            E.x = cscale(y, nr);
            continue;
        }
        const float th = uni(redC<DIM, OpAdd>(y.re * E.x.re + y.im * E.x.im));
        const float it = __builtin_amdgcn_rcpf(th);
        const cx<float> d = {fmaf(y.re, it, -E.x.re), fmaf(y.im, it, -E.x.im)};
        const float d2 = uni(redC<DIM, OpAdd>(cabs2(d)));
        const float dn = __builtin_amdgcn_sqrtf(d2);
        const float s = __builtin_amdgcn_rsqf(1.0f + d2);
        E.x = cx<float>{(E.x.re + d.re) * s, (E.x.im + d.im) * s};
        E.theta = th;
        E.dn = dn;
        E.done = false;
        if (!(dn < 3.0e38f)) return;   // not finite
        if (qb > 0.0f) {
            E.done = dn * qb * qb < 4.0e-7f * (1.0f - qb);
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

// One step of inverse iteration in residual form: with y = A x, its Rayleigh
// quotient t and r = y - t x, x becomes x - (A - sigma I)^-1 r.  The explicit
// inverse is wrong by eps |A| / mu (mu: the shift's distance from the
// eigenvalue), and so is the vector that iteration with it converges to;
// here that error multiplies r alone, and what is left is of the order of
// eps |A| / gap, as from a backward stable solver.  A = T o Gamma (HAD) or
// Gamma, from memory, four rows at a time.  Returns the squared change.
template <int DIM, bool HAD>
__device__ __forceinline__ float refine32(LdsMfma<DIM>& L, const GammaBuf& gam, const typename Acc<DIM>::type& R,
                                         const typename Acc<DIM>::type& I, int n, int col, int h, int band, float sg,
                                         EigState& E) {
    if (h == 0) {
        L.xr[col] = E.x.re;
        L.xi[col] = E.x.im;
    }
    wsync();
    float re = 0.0f, im = 0.0f;
    int o = fresh_lane(gam.offset(4 * h, col));
    const int d0 = fresh_lane(col - 4 * h);   // column - row of register 0
#pragma unroll
    for (int q = 0; q < Acc<DIM>::NV / 4; ++q) {
        const float4 xr = *(const float4*)&L.xr[8 * q + 4 * h], xi = *(const float4*)&L.xi[8 * q + 4 * h];
        const float pr[4] = {xr.x, xr.y, xr.z, xr.w}, pi[4] = {xi.x, xi.y, xi.z, xi.w};
        float m[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (HAD) {
            const float4 t = *(const float4*)&L.T[col * LdsMfma<DIM>::S + 8 * q + 4 * h];
            m[0] = t.x; m[1] = t.y; m[2] = t.z; m[3] = t.w;
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const cx<float> g = gam.at(o);
            o += (b == 3 ? 5 : 1) * n * 8;
            const bool out = band > 0 && abs(8 * q + b - d0) > band;
            const float ar = out ? 0.0f : g.re * m[b], ai = out ? 0.0f : g.im * m[b];
            re = fmaf(ar, pr[b], re);
            im = fmaf(ar, pi[b], im);
            re = fmaf(ai, pi[b], re);
            im = fmaf(-ai, pr[b], im);
        }
    }
    wsync();
    const cx<float> y = {sumH<DIM>(re), sumH<DIM>(im)};
    const float t = uni(redC<DIM, OpAdd>(y.re * E.x.re + y.im * E.x.im));
    const cx<float> r = {fmaf(-t, E.x.re, y.re), fmaf(-t, E.x.im, y.im)};
    cx<float> z = csub(r, apply32<DIM>(L, R, I, r, col, h));
    // along x the change means nothing (and is rounding, blown up by 1 / mu)
    const float cr = uni(redC<DIM, OpAdd>(E.x.re * z.re + E.x.im * z.im));
    const float ci = uni(redC<DIM, OpAdd>(E.x.re * z.im - E.x.im * z.re));
    z = cx<float>{fmaf(-cr, E.x.re, fmaf(ci, E.x.im, z.re)), fmaf(-cr, E.x.im, fmaf(-ci, E.x.re, z.im))};
    const float d2 = uni(redC<DIM, OpAdd>(cabs2(z)));
    const float s = __builtin_amdgcn_rsqf(1.0f + d2);
    E.x = cx<float>{fmaf(-sg, z.re, E.x.re) * s, fmaf(-sg, z.im, E.x.im) * s};
    return d2;
}
// Steps (nearly always one) until one changes the vector so little that what
// is left turns no component (of square m2 at least) by more than 4e-5 rad: a
// step leaves the contraction qb, and the inverse's relative error (rel: |A| /
// mu, in units of eps), of the error that it meets.  A vector that kRefines
// steps do not settle is not certified.
constexpr int kRefines = 4;
__device__ __forceinline__ float refined2(float m2, float qb, float rel) {
    const float q = qb + 8.0f * Lim<float>::eps() * rel;
    const float k = 4.0e-5f * fmaxf(1.0f - q, 0.0f) * __builtin_amdgcn_rcpf(q);
    return fmaxf(k * k * m2, 2.5e-13f);
}

// FP64 sweep of |Gamma| (diagonal stored minus 1, padding rows and columns
// zero off the diagonal and 1 on it) by pairs of pivots: the tiles (0, 0),
// (1, 0), (1, 1) become those of -|Gamma|^-1 + I.  The matrix stays symmetric,
// so the pivots of the first tile row update the tiles on and right of the
// diagonal, those of the second the tiles on and left of it, with tile (0, 1)
// transposed into (1, 0) through LDS in between: three MFMAs a pair, not
// four.  Returns whether every pivot was positive; near: a pivot up to the
// first one that is not positive lay within kCertPivotMin of 0.
template <int K, int NB>
__device__ __forceinline__ void sweep64_rows(mf64x4 (&M)[NB][NB], int n, const double (&al)[2], const double (&be)[2],
                                             const double (&ga)[2], bool& ok, bool& near) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int s = 0; s < 4; s += 2) {
            if (16 * K + 4 * r + s >= fresh(n) || !ok) continue;
            const double x = M[K][K][r];
            const double d00 = lane_f64(x, 16 * s + 4 * r + s) + 1.0;
            const double d01 = lane_f64(x, 16 * s + 4 * r + s + 1);
            const double d11 = lane_f64(x, 16 * (s + 1) + 4 * r + s + 1) + 1.0;
            const double det = fma(-d01, d01, d00 * d11);   // the second pivot is det / d00
            if (!(fmin(det, d00 * d00) >= kCertPivotMin * d00) || !(d00 > 0.0)) {   // rarely
                near = near | (fabs(d00) < kCertPivotMin) | (fabs(det) < kCertPivotMin * d00);
                ok = (d00 > 0.0) & (det > 0.0);
            }
            // W = -D^-1 X for the pair's rows X, zero in the other two rows of
            // the register: the 4x4x4 MFMA takes A[i][k] in lanes
            // i + 4 block + 16 k, and X and W as they lie in the tiles
            const double num = fma(ga[s / 2], d00, fma(be[s / 2], d01, al[s / 2] * d11));
            const double ca = num * fast_rcp(det);
            double b[NB], w[NB];
#pragma unroll
            for (int J = 0; J < NB; ++J) {
                b[J] = M[K][J][r];
                asm("" : "+v"(b[J]));   // its own registers: the tile is overwritten below
                w[J] = __builtin_amdgcn_mfma_f64_4x4x4f64(ca, b[J], 0.0, 0, 0, 0);
            }
            M[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[0], b[0], M[0][0], 0, 0, 0);
            if constexpr (NB == 2) {
                M[K][1 - K] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[K], b[1 - K], M[K][1 - K], 0, 0, 0);
                M[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[1], b[1], M[1][1], 0, 0, 0);
            }
        }
}
template <int DIM>
__device__ __forceinline__ bool sweep64(LdsMfma<DIM>& L, mf64x4 (&M)[DIM / 16][DIM / 16], int n, int lane, bool& near) {
    bool ok = true;
    near = false;
    const int q = lane >> 4, i = lane & 3;
    double al[2], be[2], ga[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {   // this lane's entry of -adj(D) in terms of d11, d01, d00
        const int s = 2 * k;
        al[k] = i == s && q == s ? -1.0 : 0.0;
        ga[k] = i == s + 1 && q == s + 1 ? -1.0 : 0.0;
        be[k] = (i == s && q == s + 1) || (i == s + 1 && q == s) ? 1.0 : 0.0;
    }
    sweep64_rows<0, DIM / 16>(M, n, al, be, ga, ok, near);
    if constexpr (DIM == 32) {
        double* X = (double*)L.T;   // 16 x 16, rows 17 apart
#pragma unroll
        for (int r = 0; r < 4; ++r) X[(4 * r + q) * 17 + (lane & 15)] = M[0][1][r];
        wsync();
#pragma unroll
        for (int r = 0; r < 4; ++r) M[1][0][r] = X[(lane & 15) * 17 + 4 * r + q];
        wsync();
        sweep64_rows<1, 2>(M, n, al, be, ga, ok, near);
    }
    return ok;
}

// |Gamma| into the FP64 tiles (diagonal stored minus 1 = 0, also in the
// padding); false when an entry is not finite.
template <int NB>
__device__ __forceinline__ bool load_abs64(const GammaBuf& gam, int n, int lane, mf64x4 (&M)[NB][NB]) {
    float sum = 0.0f;
    const int o0 = gam.offset(lane >> 4, lane & 15), o1 = gam.offset(lane >> 4, 16 + (lane & 15));
    const int dr = (lane & 15) - (lane >> 4);   // 4 r on the diagonal
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
        for (int J = 0; J < NB; ++J)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const cx<float> g = gam.at((J ? o1 : o0) + (16 * K + 4 * r) * n * 8);
                float v = __builtin_amdgcn_sqrtf(g.re * g.re + g.im * g.im);
                if (K == J && dr == 4 * r) v = 0.0f;
                sum += v;
                M[K][J][r] = (double)v;
            }
    return __all(sum < 3.0e38f);
}

// I - M -> |Gamma|^-1 in FP32 rows in LDS (tile (0, 1) from (1, 0))
template <int DIM>
__device__ __forceinline__ void inverse_to_lds(LdsMfma<DIM>& L, const mf64x4 (&M)[DIM / 16][DIM / 16], int lane) {
    constexpr int S = LdsMfma<DIM>::S;
    const int q = lane >> 4, c = lane & 15, dr = c - q;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + q;
        const double one = dr == 4 * r ? 1.0 : 0.0;
        L.T[row * S + c] = (float)(one - M[0][0][r]);
        if constexpr (DIM == 32) {
            L.T[(16 + row) * S + 16 + c] = (float)(one - M[1][1][r]);
            const float m = -(float)M[1][0][r];
            L.T[(16 + row) * S + c] = m;
            L.T[c * S + 16 + row] = m;
        }
    }
}

// One pixel on the 64 lanes of a wave.
template <int MODE, int DIM>
__device__ __forceinline__ void solve_mfma_pixel(const SolveArgs& a, LdsMfma<DIM>& L, int lane, int np,
                                                 const GammaBuf& gam, long long pix) {
    typedef typename Acc<DIM>::type acc;
    constexpr int NV = Acc<DIM>::NV, S = LdsMfma<DIM>::S;
    const int n = a.n, col = lane & (DIM - 1), h = lane / DIM;
    const bool in = col < n;
    // register of this lane's diagonal entry
    const int vd0 = ((col >> 2) & (64 / DIM - 1)) == h ? (DIM == 32 ? 4 * (col >> 3) : 0) + (col & 3) : -1;
    const bool stbas = a.method == FRINGE_METHOD_STBAS && MODE == MODE_EVD;
    float code = 0.0f;
    bool unc = false;
    bool inv = MODE != MODE_EVD;   // matrix: H (smallest eigenvalue), else Gamma (largest)
    EigState E;
    E.x = cx<float>{0.0f, 0.0f};

    const bool act = np >= 0;
    if (act) {
        if constexpr (MODE == MODE_MLE) {
            // smallest eigenvalue of Gamma at least 1e-6, by a margin
            // (Gamma has unit diagonal: its norm is at most n)
            acc R, I;
            load_gamma32<DIM>(gam, n, col, h, R, I);
            const float s = 1.0e-6f + kCertThrMargin * Lim<float>::eps() * (float)n;
            float sum = 0.0f;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                sum += fabsf(R[v]) + fabsf(I[v]);
                if (v == vd0) R[v] = -s;   // 1 - s, stored minus 1
            }
            if (!__all(sum < 3.0e38f)) {
                code = -1.0f;
            } else {
                int neg;
                int near;
                sweep32(R, I, n, lane, neg, near);
                unc = neg != 0;
            }
        }
        if constexpr (MODE != MODE_EVD) {
            if (code == 0.0f && !unc) {
                mf64x4 M[DIM / 16][DIM / 16];
                const bool fin = load_abs64<DIM / 16>(gam, n, lane, M);
                if (!fin) {
                    code = -1.0f;
                } else {
                    bool near;
                    const bool pd = sweep64<DIM>(L, M, n, lane, near);
                    unc = near;
                    if (MODE == MODE_EMI) inv = pd;   // else the EVD fallback
                    else unc = unc || !pd;
                    if (inv) inverse_to_lds<DIM>(L, M, lane);
                    wsync();
                    if constexpr (MODE == MODE_MLE) {
                        // |Gamma| - 1e-6 I is positive definite when its
                        // smallest eigenvalue, at least 1 / trace(inverse), is
                        const float tr = redC<DIM, OpAdd>(in ? L.T[col * S + col] : 0.0f);
                        unc = unc || !(uni(tr) < 1.0e5f);
                    }
                }
            }
        }
    }

    // ---- the eigenpair ----
    if (act && code == 0.0f && !unc) {
        // start: the phases of the middle column
        const cx<float> g = gam.at(gam.offset(n >> 1, col));
        const float g2 = cabs2(g);
        const float is = __builtin_amdgcn_rsqf((float)n);
        const float w = g2 > 0.0f ? __builtin_amdgcn_rsqf(g2) * is : 0.0f;
        E.x = cx<float>{g.re * w, -g.im * w};
        if (in && !(g2 > 0.0f)) E.x.re = is;
        float sigma = 1.0f, sg = 1.0f, tn = 1.0f;
        const float dg = inv ? (in ? L.T[col * S + col] : 0.0f) : 1.0f;
        if (!inv) {
            sg = -1.0f;
            if constexpr (MODE == MODE_EMI) {   // Gamma = T o Gamma
                for (int e = lane; e < DIM * S; e += 64) L.T[e] = 1.0f;
                wsync();
            }
            acc R, I;
            load_gamma32<DIM>(gam, n, col, h, R, I);
            float f2 = 0.0f, sum = 0.0f;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if (stbas && abs(Acc<DIM>::row(v, 0) - fresh_lane(col - 4 * h)) > a.bw) {
                    R[v] = 0.0f;
                    I[v] = 0.0f;
                }
                f2 = fmaf(R[v], R[v], fmaf(I[v], I[v], f2));
            }
            sum = uni(sumH<DIM>(redC<DIM, OpAdd>(f2)));
            if (MODE == MODE_EVD && !(sum < 3.0e38f)) code = -6.0f;
            if (code == 0.0f) {
                float rho = 1.0f, dn = 1.0f;
                for (int k = 0; k < 3; ++k) {
                    const cx<float> y = apply32<DIM>(L, R, I, E.x, col, h);
                    rho = uni(redC<DIM, OpAdd>(y.re * E.x.re + y.im * E.x.im));
                    const float it = __builtin_amdgcn_rcpf(rho);
                    const cx<float> d = {y.re * it - E.x.re, y.im * it - E.x.im};
                    dn = uni(redC<DIM, OpAdd>(cabs2(d)));
                    const float s = __builtin_amdgcn_rsqf(1.0f + dn);
                    E.x = cx<float>{(E.x.re + d.re) * s, (E.x.im + d.im) * s};
                }
                // the residual of the last vector but one bounds the distance
                // to an eigenvalue; the largest lies above the quotient
                sigma = rho + rho * fmaxf(__builtin_amdgcn_sqrtf(dn), 0.02f);
                const float m2 = sum * a.inv_n - 1.0f;
                tn = 1.0f + __builtin_amdgcn_sqrtf(fmaxf(m2, 0.0f) * (float)(n - 1));
            }
        }
        bool certified = false, checking = false, close = false;
        float lam = 0.0f, delta = 0.0f;
        if (code == 0.0f)
            for (int att = 0; att < 6; ++att) {
                const int vd = fresh_lane(vd0);
                // ---- B = +-(A - sigma I), diagonal minus 1 ----
                const float off = in ? sg * (dg - sigma) - 1.0f : 0.0f;
                acc R, I;
                load_gamma32<DIM>(gam, n, col, h, R, I);
                float f2 = 0.0f;
                if (inv) {
#pragma unroll
                    for (int q = 0; q < NV / 4; ++q) {
                        const float4 m = *(const float4*)&L.T[col * S + 8 * q + 4 * h];
                        const float mm[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const int v = 4 * q + b;
                            R[v] *= mm[b];
                            I[v] *= mm[b];
                            if (v != vd) f2 = fmaf(R[v], R[v], fmaf(I[v], I[v], f2));
                            else R[v] = off;
                        }
                    }
                    if (att == 0) {
                        // |H| <= m + s sqrt(n - 1) with m the mean and s the
                        // deviation of the eigenvalues (Wolkowicz and Styan)
                        const float tr = uni(redC<DIM, OpAdd>(dg)) * a.inv_n;
                        const float ff = uni(sumH<DIM>(redC<DIM, OpAdd>(f2 + (vd >= 0 ? dg * dg : 0.0f)))) * a.inv_n;
                        tn = tr + __builtin_amdgcn_sqrtf(fmaxf(ff - tr * tr, 0.0f) * (float)(n - 1));
                        if (!(tn < 3.0e38f)) break;   // H not finite: the FP64 path decides
                    }
                } else {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const bool out = stbas && abs(Acc<DIM>::row(v, 0) - fresh_lane(col - 4 * h)) > a.bw;
                        R[v] = out ? 0.0f : -R[v];
                        I[v] = out ? 0.0f : -I[v];
                        if (v == vd) R[v] = off;
                    }
                }
                int neg;
                int near;
                sweep32(R, I, n, lane, neg, near);
                if (checking) {   // B's shift lies delta past the eigenvalue: only that one below it
                    certified = neg <= 1 && near >= 1700;
                    break;
                }
                if (neg > 1) {   // the shift passed a second eigenvalue
                    if (inv) sigma = sigma > 0.5f ? 0.5f * sigma : 0.0f;
                    else sigma = sigma * 1.15f;
                    continue;
                }
                iterate32<DIM>(L, R, I, col, h, 0.0f, E);
                const float mu = __builtin_amdgcn_rcpf(E.theta);
                lam = sigma + sg * mu;
                if (!(fabsf(lam) < 3.0e38f)) break;
                if (!E.done) {
                    // eigenvalues of B: mu, and the next one at |mu| / q on the
                    // far side; move the shift next to the first
                    const float q = E.q > 0.0f ? fminf(fmaxf(E.q, 1.0e-3f), 0.98f) : 0.98f;
                    const float gap = fabsf(mu) / q - mu;
                    const float e = fminf(E.dn * q / (1.0f - q), 1.0f);
                    sigma += sg * (mu - (e * e + 0.15f) * gap);
                    continue;
                }
                // ---- certification ----
                const float m2 = redC<DIM, OpMin>(in ? cabs2(E.x) : 3.0e38f);
                delta = cert_eps(inv, a.cert_h, a.cert_g, tn) * tn * __builtin_amdgcn_rsqf(uni(m2));
                if (!(delta <= tn)) break;
                // Frobenius norm of the inverse: its other eigenvalues'
                // squares sum to S2, so none of them exceeds sqrt(S2)
                float f = 0.0f;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const float x = v == vd ? 1.0f - R[v] : R[v];
                    f = fmaf(x, x, fmaf(I[v], I[v], f));
                }
                if (vd >= 0 && !in) f -= 1.0f;   // padding: R = 0 on the diagonal
                f = uni(sumH<DIM>(redC<DIM, OpAdd>(f)));
                const float s2 = fmaxf(f - E.theta * E.theta, 0.0f) + 4.0e-6f * f;
                const float t = mu + delta;
                const bool side = neg == 0 ? E.theta > 0.0f : E.theta < 0.0f;
                if (!side) break;
                // the contraction is at most qb: the error left by the last step
                const float qb = __builtin_amdgcn_sqrtf(s2) * fabsf(mu);
                bool conv = qb < 0.8f;
                if (conv && E.dn * qb * qb > 4.0e-7f * (1.0f - qb)) {
                    iterate32<DIM>(L, R, I, col, h, qb, E);
                    conv = E.done;
                }
                // a shift inside the spectrum: small pivots would have cost accuracy
                if (neg != 0 && near < kNearInside && !close) conv = false;
                certified = conv && (t <= 0.0f || s2 * t * t < 1.0f);
                if (certified || (conv && close)) {
                    const float most = refined2(uni(m2), qb, tn * fabsf(E.theta));
                    float d2 = 1.0f;
                    for (int k = 0; k < kRefines && d2 > most; ++k)
                        d2 = refine32<DIM, MODE != MODE_EVD>(L, gam, R, I, n, col, h, stbas ? a.bw : 0, sg, E);
                    if (!(d2 <= most)) certified = conv = false;
                }
                if (certified) break;
                // the next eigenvalue as the measured contraction places it is
                // too close for any certificate: the FP64 path's pixel
                if (E.q > 0.02f && E.dq > 4.0e-6f && fabsf(mu) * __builtin_amdgcn_rcpf(E.q) - mu < 0.7f * delta) break;
                if (!close) {   // once more from a quarter of the distance away
                    close = true;
                    sigma = lam - sg * 0.25f * delta;
                    continue;
                }
                if (!conv) break;
                checking = true;
                sigma = lam + sg * delta;
            }
        if constexpr (MODE == MODE_EVD) unc = unc || !(lam >= 1.0e-6f + kCertThrMargin * Lim<float>::eps() * tn);
        if constexpr (MODE == MODE_MLE) unc = unc || !(lam >= 1.0e-6f + kCertThrMargin * Lim<float>::eps() * tn);
        unc = code == 0.0f && (unc || !certified);
    }

    if (act && unc) {   // the FP64 re-solve writes every output of the pixel
        if (lane == 0) {
            const int e = atomicAdd(a.cert_count, 1);
            if (e < a.cert_cap) a.cert_list[e] = (int)pix;
        }
        return;
    }
    const bool ok = act && code == 0.0f;
    if (!ok) {
        if (lane < n) a.phase[(long long)lane * a.npx + pix] = make_float2(0.0f, 0.0f);
        if (lane == 0) {
            a.tcorr[pix] = code;
            a.comp[pix] = make_float2(0.0f, 0.0f);
        }
        return;
    }

    // ---- referenced phases (evd.cpp:738-749) ----
    const cx<float> vref = {lane_f32(E.x.re, a.ref), lane_f32(E.x.im, a.ref)};
    const cx<float> uv = cmulc(E.x, vref);
    const float u2 = cabs2(uv);
    float ur = __builtin_amdgcn_rsqf(u2);
    ur = ur * fmaf(-0.5f * u2 * ur, ur, 1.5f);   // one Newton step
    cx<float> o = cscale(uv, ur);
    if (__any(in && !(u2 > 1.0e-36f))) {   // a zero, or nearly, component
        bool okr, oku, okv;
        const cx<float> cref = unit_or(cconj(vref), cx<float>{1.0f, 0.0f}, okr);
        const cx<float> u = unit_or(uv, cx<float>{0.0f, 0.0f}, oku);
        o = oku ? u : (okr ? cref : unit_or(E.x, cx<float>{1.0f, 0.0f}, okv));
    }
    if (col == a.ref) o = cx<float>{1.0f, 0.0f};
    if (lane < n) a.phase[(long long)lane * a.npx + pix] = make_float2(o.re, o.im);
    // ---- compressed SLC (evd.cpp:755-762) ----
    cx<double> cs = {0.0, 0.0};
    if (col >= a.ref && in) {
        const float2 z = a.slc[(long long)col * a.npx + pix];
        cs.re = (double)(z.x * o.re + z.y * o.im);
        cs.im = (double)(z.y * o.re - z.x * o.im);
    }
    cs = cx<double>{redC<DIM, OpAdd>(cs.re), redC<DIM, OpAdd>(cs.im)};
    // ---- temporal coherence (evd.cpp:770-786): sum over i < j (j <= i + bw
    // for STBAS) of exp(i (arg Gamma_ij - arg o_i + arg o_j)) ----
    if (h == 0) {
        L.xr[col] = in ? o.re : 0.0f;
        L.xi[col] = in ? o.im : 0.0f;
    }
    wsync();
    float xr[NV], xi[NV];
    row_values<DIM>(L, h, xr, xi);
    acc R, I;
    load_gamma32<DIM>(gam, n, col, h, R, I);
    float tr = 0.0f, ti = 0.0f;
    const int rb = stbas ? col - a.bw : 0;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int row = Acc<DIM>::row(v, h);
        float rs = __builtin_amdgcn_rsqf(fmaf(R[v], R[v], I[v] * I[v]));
        rs = row < col ? rs : 0.0f;
        if (stbas && row < rb) rs = 0.0f;
        const float pr = R[v] * rs, pi = I[v] * rs;
        tr = fmaf(pr, xr[v], fmaf(pi, xi[v], tr));   // Gamma_ij / |Gamma_ij| conj(o_i)
        ti = fmaf(pi, xr[v], fmaf(-pr, xi[v], ti));
    }
    if (__any(in && !(fabsf(tr) < 3.0e38f))) {   // a zero entry, whose phase counts as 0
        tr = 0.0f;
        ti = 0.0f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int row = Acc<DIM>::row(v, h);
            const float g2 = fmaf(R[v], R[v], I[v] * I[v]);
            const bool use = row < col && !(stbas && row < rb), z = !(g2 > 0.0f);
            const float rs = use ? __builtin_amdgcn_rsqf(g2) : 0.0f;
            const float pr = z ? (use ? 1.0f : 0.0f) : R[v] * rs, pi = z ? 0.0f : I[v] * rs;
            tr = fmaf(pr, xr[v], fmaf(pi, xi[v], tr));
            ti = fmaf(pi, xr[v], fmaf(-pr, xi[v], ti));
        }
    }
    float sr = tr * o.re - ti * o.im, si = tr * o.im + ti * o.re;
    if (!in) {
        sr = 0.0f;
        si = 0.0f;
    }
    sr = sumH<DIM>(redC<DIM, OpAdd>(sr));
    si = sumH<DIM>(redC<DIM, OpAdd>(si));
    if (lane == 0) {
        // |sum| / pairs in double: rsq refined by one Newton step
        const double s2 = (double)sr * (double)sr + (double)si * (double)si;
        double rs = __builtin_amdgcn_rsq(s2);
        rs = rs * fma(-0.5 * s2 * rs, rs, 1.5);
        a.tcorr[pix] = (float)((s2 > 0.0 ? s2 * rs : 0.0) * a.inv_pairs);
        a.comp[pix] = make_float2((float)(cs.re * a.inv_comp), (float)(cs.im * a.inv_comp));
    }
}

// WPB waves (pixels) per workgroup; slots last-first (the coherence matrices
// the Gram wrote last are the ones still in the last-level cache).
template <int MODE, int DIM, int WPB>
__global__ __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(DIM == 32 ? 4 : 6))) void solve_mfma_kernel(SolveArgs a) {
    __shared__ LdsMfma<DIM> sm[WPB];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int slot = a.slots - 1 - ((int)blockIdx.x * WPB + w);
    if (slot < 0) return;
    const int np = a.npix[slot];
    const cx<float>* gam = (const cx<float>*)a.gamma + (size_t)slot * a.n * a.n;
    solve_mfma_pixel<MODE, DIM>(a, sm[w], lane, np, GammaBuf(gam, a.n), a.first + slot);
}

}  // namespace fringe
