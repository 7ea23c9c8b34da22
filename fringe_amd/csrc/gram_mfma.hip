// gram_mfma.hip -- masked-neighbourhood coherence on the MFMA units (gfx950).
//
// For a pixel with compacted SHP neighbour list k = 1..K (positions whose
// mask bit is set and which lie inside the tile, evd.cpp:530-564), the
// complex Gram G = sum_k z_k z_k^H is computed as the real Gram P = Y^T Y of
// Y = [Re z | Im z] (K x 2n):
//     Re G_ij = P(re_i, re_j) + P(im_i, im_j)
//     Im G_ij = P(im_i, re_j) - P(re_i, im_j)
// Each sample is split once into a 16-bit hi + lo pair (hi = h(x), lo =
// h(x - hi)) and P is accumulated in FP32 over hi*hi + hi*lo + lo*hi, by
// v_mfma_f32_16x16x32_{f16,bf16} in the staged kernel and by 32x32x16 in the
// gathering ones.
//   * fp16 (default): every date is first scaled by an exact power of two so
//     that its largest |Re|, |Im| over the tile lies in [2^14, 2^15); the pair
//     then carries ~22 significant bits.  The coherence
//     Gamma_ij = G_ij / sqrt(G_ii G_jj) is invariant to per-date scaling, so
//     the scale never has to be undone.
//   * bf16: the pair carries ~16 bits and keeps the FP32 exponent range, so
//     no scaling is applied.
//
// Data flow:
//   pack_hilo : the band-planar stack slc[t][row][col] is rewritten once as
//               position-major packed words pk[pixel][re_0, im_0, re_1,
//               im_1, ...] with (hi | lo << 16); one extra all-zero record at
//               index rows*cols pads neighbour lists.
//   gram_mfma_lds (up to 64 dates) : the records a pixel tile's windows share
//               are staged in LDS; one wave per pixel at a time.
//   gram_mfma : where no tile fits LDS; one wave per pixel at a time.  The
//               wave compacts the mask into a list of pixel indices (padded
//               to a multiple of 16) in LDS; per 16 positions lane l gathers
//               component (l % 32) of 8 positions for every 32-wide component
//               block -- lanes 0..31 read one contiguous 128-byte record
//               slice, lanes 32..63 another -- and issues 3 MFMAs per block
//               pair.  The upper
//               block triangle of P is folded into Gamma (the transposed
//               cross block goes through a per-wave LDS scratch) and written.
//               Above 32 dates (gram_mfma_pairs) the wave walks the pairs of
//               32-date blocks one at a time instead of holding every block.
#include <algorithm>

#include "device_common.hpp"
#include "engine_internal.hpp"
#include "fringe_amd.h"

namespace fringe {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;

// Round-to-nearest-even float -> bf16 bits (finite input).
__device__ inline uint32_t bf16_rne(float x) {
    const uint32_t u = __float_as_uint(x);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ inline uint32_t split_hi_lo_bf16(float x) {
    const uint32_t hi = bf16_rne(x);
    const float rest = x - __uint_as_float(hi << 16);
    const uint32_t lo = bf16_rne(rest);
    return hi | (lo << 16);
}
__device__ inline uint32_t split_hi_lo_f16(float x) {
    const _Float16 hi = (_Float16)x;
    const _Float16 lo = (_Float16)(x - (float)hi);
    return (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
}

// ---- per-date largest |Re|, |Im| over the tile ----------------------------
// Non-negative floats order like their bit patterns, so the maximum is kept
// as an unsigned word with atomicMax.
__global__ void date_absmax_clear(uint32_t* dmax, int n) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dmax[t] = 0u;
}
// NT threads; one workgroup per date writes its maximum, several take theirs
// together over a cleared word.
template <int NT>
__global__ __launch_bounds__(NT) void date_absmax(const float2* __restrict__ slc, long long npx,
                                                  uint32_t* __restrict__ dmax) {
    const int t = blockIdx.y;
    const float2* __restrict__ band = slc + (long long)t * npx;
    const long long stride = (long long)gridDim.x * blockDim.x;
    long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    // Largest finite |Re|, |Im|: an infinite or NaN sample makes only the
    // coherence of the windows that hold it non-finite (as in FP64), and must
    // not take the scale of the whole date with it.  Four independent loads
    // in flight per thread; the maximum does not depend on the order.
    auto fin_abs = [](float2 z) {
        const float a = fmaxf(fabsf(z.x), fabsf(z.y));   // NaN parts dropped
        return (a < INFINITY && z.x == z.x && z.y == z.y) ? a : 0.0f;
    };
    for (; p + 3 * stride < npx; p += 4 * stride) {
        float2 z[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) z[k] = band[p + k * stride];
#pragma unroll
        for (int k = 0; k < 4; ++k) m = fmaxf(m, fin_abs(z[k]));
    }
    for (; p < npx; p += stride) m = fmaxf(m, fin_abs(band[p]));
    for (int o = 32; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    // one atomic per workgroup: every date's word shares a cache line, and
    // atomics on one line serialise
    __shared__ float wm[NT / 64];
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 1; k < NT / 64; ++k) m = fmaxf(m, wm[k]);
        if (gridDim.x == 1) dmax[t] = __float_as_uint(m);
        else atomicMax(dmax + t, __float_as_uint(m));
    }
}
// Power-of-two exponent k with max * 2^k in [2^14, 2^15); 0 when the date is
// all zero or not finite.
__device__ inline int date_scale_exp(uint32_t bits) {
    const float m = __uint_as_float(bits);
    if (!(m > 0.0f) || !isfinite(m)) return 0;
    int e;
    frexpf(m, &e);          // m in [2^(e-1), 2^e)
    return min(15 - e, 126);
}

// ---- pack: [t][pixel] complex64 -> [pixel][2n] (hi|lo) words -------------
// 64 pixels per workgroup; the band-planar rows are read coalesced and the
// records written contiguously through an LDS transpose.
template <bool F16>
__global__ __launch_bounds__(256) void pack_hilo(const float2* __restrict__ slc, int n,
                                                 long long npx, const uint32_t* __restrict__ dmax,
                                                 uint32_t* __restrict__ pk, int* __restrict__ count) {
    if (count && blockIdx.x == 0 && threadIdx.x == 0) *count = 0;   // the run's list of uncertified pixels
    extern __shared__ uint32_t st[];   // [64][2n]
    const long long p0 = (long long)blockIdx.x * 64;
    const int CS = 2 * n;
    for (int e = threadIdx.x; e < 64 * n; e += blockDim.x) {
        const int t = e / 64, i = e % 64;
        const long long p = p0 + i;
        float2 z = make_float2(0.0f, 0.0f);
        if (p < npx) z = slc[(long long)t * npx + p];
        if (F16) {
            const int k = date_scale_exp(dmax[t]);
            st[i * CS + 2 * t] = split_hi_lo_f16(ldexpf(z.x, k));
            st[i * CS + 2 * t + 1] = split_hi_lo_f16(ldexpf(z.y, k));
        } else {
            st[i * CS + 2 * t] = split_hi_lo_bf16(z.x);
            st[i * CS + 2 * t + 1] = split_hi_lo_bf16(z.y);
        }
    }
    __syncthreads();
    const long long words = (long long)min((long long)64, npx - p0) * CS;
    for (long long e = threadIdx.x; e < words; e += blockDim.x) pk[p0 * CS + e] = st[e];
    if (blockIdx.x == 0)
        for (int e = threadIdx.x; e < CS; e += blockDim.x) pk[npx * CS + e] = 0u;
}

// The staged kernel reads a pixel's mask words from lanes 0..15, two words
// per 64-position pass: windows of up to 512 positions.
constexpr int kStageWords = 16;

struct MfmaArgs {
    const uint32_t* pk;   // packed records, [rows*cols + 1][n][re, im]
    const uint32_t* wts;
    int rows, cols, n, Nx, Ny, nul, min_nb;
    int row0;             // first output row of this chunk
    int chunk_rows;
    int TH, TW;           // output pixels per workgroup
    float* gamma;         // [slots][n][n] complex float, interleaved
    int* npix;            // [slots]
    int list_cap;         // ints per wave list
};

// 32x32 accumulator layout: lane l, element v holds C[row][col] with
// col = l % 32 and row = 8*(v/4) + 4*(l/32) + (v%4).
__device__ inline int acc_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

template <int NBH> struct TileIdx {
    static constexpr int NB = 2 * NBH;
    // (bi, bj), bi <= bj < NB, in row-major upper order
    static __device__ constexpr int idx(int bi, int bj) {
        return bi * NB - (bi * (bi - 1)) / 2 + (bj - bi);
    }
    static constexpr int count = NB * (NB + 1) / 2;
};

__device__ inline void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool F16> struct Frag;
template <> struct Frag<true> {
    typedef f16x8 type;
    static __device__ inline f32x16 mfma(type a, type b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};
template <> struct Frag<false> {
    typedef bf16x8 type;
    static __device__ inline f32x16 mfma(type a, type b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

template <int NBH, int WAVES, bool F16>
__global__ __launch_bounds__(64 * WAVES) void gram_mfma(MfmaArgs a) {
    typedef typename Frag<F16>::type frag_t;
    constexpr int NB = 2 * NBH;
    constexpr int NT = TileIdx<NBH>::count;
    extern __shared__ __align__(16) char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const size_t wbytes = (size_t)a.list_cap * 4 + 32 * 33 * 4 + 64 * NBH * 4;
    int* list = (int*)(smem + (size_t)wave * wbytes);
    float* xs = (float*)(list + a.list_cap);   // 32 x 33 transpose scratch
    float* dg = xs + 32 * 33;                  // diagonal of Re G

    const int n = a.n, Nx = a.Nx, Ny = a.Ny;
    const int CS = 2 * n;
    const int npx_zero = a.rows * a.cols;      // index of the all-zero record
    const int R0 = a.row0 + blockIdx.y * a.TH, C0 = blockIdx.x * a.TW;
    const int row_end = a.row0 + a.chunk_rows;
    const int Wx = 2 * Nx + 1, Wn = (2 * Ny + 1) * Wx;
    const int m = lane & 31, half = lane >> 5;

    uint32_t coff[NB];
    bool cval[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int date = 32 * (b % NBH) + m;
        cval[b] = date < n;
        coff[b] = cval[b] ? (uint32_t)(2 * date + (b < NBH ? 0 : 1)) : 0u;
    }

    for (int pid = wave; pid < a.TH * a.TW; pid += WAVES) {
        const int r = R0 + pid / a.TW, c = C0 + pid % a.TW;
        if (r >= row_end || r >= a.rows || c >= a.cols) continue;   // wave-uniform
        const long long pix = (long long)r * a.cols + c;
        const int slot = (r - a.row0) * a.cols + c;
        const uint32_t* w = a.wts + pix * a.nul;
        const bool cen = shp_get(w, shp_flat(0, 0, Nx, Ny));

        // ---- neighbour list ----
        int cnt = 0;
        for (int b0 = 0; b0 < Wn; b0 += 64) {
            const int f = b0 + lane;
            bool take = false;
            int q = 0;
            if (cen && f < Wn) {
                const int rr = r + f / Wx - Ny, cc = c + f % Wx - Nx;
                if (rr >= 0 && rr < a.rows && cc >= 0 && cc < a.cols && shp_get(w, f)) {
                    take = true;
                    q = rr * a.cols + cc;
                }
            }
            const uint64_t bal = __ballot(take);
            if (take) {
                const uint64_t below = (lane == 0) ? 0ull : (bal & ((~0ull) >> (64 - lane)));
                list[cnt + __popcll(below)] = q;
            }
            cnt += __popcll(bal);
        }
        if (!(cen && cnt >= a.min_nb)) {
            if (lane == 0) a.npix[slot] = -1;
            continue;
        }
        const int steps = (cnt + 15) >> 4;
        for (int e = cnt + lane; e < steps * 16; e += 64) list[e] = npx_zero;
        wave_sync_lds();

        // ---- MFMA accumulation ----
        f32x16 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

        for (int s = 0; s < steps; ++s) {
            const int* lp = list + 16 * s + 8 * half;
            uint32_t base[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) base[e] = (uint32_t)lp[e] * (uint32_t)CS;
            frag_t fh[NB], fl[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                uint32_t wv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[e] = a.pk[base[e] + coff[b]];   // valid address for every lane
#pragma unroll
                for (int e = 0; e < 8; ++e) wv[e] = cval[b] ? wv[e] : 0u;
                u32x4 hv, lv;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hv[e] = __builtin_amdgcn_perm(wv[2 * e + 1], wv[2 * e], 0x05040100u);
                    lv[e] = __builtin_amdgcn_perm(wv[2 * e + 1], wv[2 * e], 0x07060302u);
                }
                fh[b] = __builtin_bit_cast(frag_t, hv);
                fl[b] = __builtin_bit_cast(frag_t, lv);
            }
#pragma unroll
            for (int bi = 0; bi < NB; ++bi)
#pragma unroll
                for (int bj = bi; bj < NB; ++bj) {
                    f32x16& C = acc[TileIdx<NBH>::idx(bi, bj)];
                    C = Frag<F16>::mfma(fh[bi], fh[bj], C);
                    C = Frag<F16>::mfma(fh[bi], fl[bj], C);
                    C = Frag<F16>::mfma(fl[bi], fh[bj], C);
                }
        }

        // ---- fold P into Gamma ----
#pragma unroll
        for (int I = 0; I < NBH; ++I) {
            const f32x16& A0 = acc[TileIdx<NBH>::idx(I, I)];
            const f32x16& A1 = acc[TileIdx<NBH>::idx(NBH + I, NBH + I)];
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (acc_row(v, lane) == m) dg[32 * I + m] = A0[v] + A1[v];
        }
        float* gout = a.gamma + (size_t)slot * n * n * 2;
#pragma unroll
        for (int I = 0; I < NBH; ++I)
#pragma unroll
            for (int J = I; J < NBH; ++J) {
                const f32x16& X = acc[TileIdx<NBH>::idx(J, NBH + I)];   // P(re_J, im_I)
                wave_sync_lds();
#pragma unroll
                for (int v = 0; v < 16; ++v) xs[acc_row(v, lane) * 33 + m] = X[v];
                wave_sync_lds();
                const f32x16& RR = acc[TileIdx<NBH>::idx(I, J)];
                const f32x16& II = acc[TileIdx<NBH>::idx(NBH + I, NBH + J)];
                const f32x16& RI = acc[TileIdx<NBH>::idx(I, NBH + J)];
                const int j = 32 * J + m;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int il = acc_row(v, lane);
                    const int i = 32 * I + il;
                    if (i >= n || j >= n || i > j) continue;
                    float gr = 1.0f, gi = 0.0f;
                    if (i != j) {
                        const float re = RR[v] + II[v];
                        const float im = xs[m * 33 + il] - RI[v];   // P(im_i, re_j) - P(re_i, im_j)
                        const float sc = rsqrtf(dg[i] * dg[j]);
                        gr = re * sc;
                        gi = im * sc;
                    }
                    gout[2 * ((size_t)i * n + j)] = gr;
                    gout[2 * ((size_t)i * n + j) + 1] = gi;
                    if (i != j) {
                        gout[2 * ((size_t)j * n + i)] = gr;
                        gout[2 * ((size_t)j * n + i) + 1] = -gi;
                    }
                }
            }
        if (lane == 0) a.npix[slot] = cnt;
        wave_sync_lds();
    }
}

// 64 < n <= 128, and 33..64 where nothing can be staged: the wave of a pixel walks the date-block pairs (I, J),
// I <= J < nb = ceil(n / 32), diagonal pairs first.  Per pair it keeps the
// four 32 x 32 real products P(re_I, re_J), P(im_I, im_J), P(re_I, im_J),
// P(im_I, re_J) (64 accumulator registers whatever n; 12 MFMAs per 16
// positions) and writes Gamma block (I, J) and its mirror; Re G_ii of the
// diagonal pairs (per-wave LDS) normalises the later ones.  Each position's
// (re, im) word pair of a date is one 8-byte load, and records are addressed
// with 64-bit offsets (2n words per record exceed 32-bit word offsets on
// large tiles).
template <int WAVES, bool F16>
__global__ __launch_bounds__(64 * WAVES) void gram_mfma_pairs(MfmaArgs a) {
    typedef typename Frag<F16>::type frag_t;
    extern __shared__ __align__(16) char smem[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const size_t wbytes = (size_t)a.list_cap * 4 + 128 * 4;
    int* list = (int*)(smem + (size_t)wave * wbytes);
    float* dg = (float*)(list + a.list_cap);   // Re G_ii of the pixel, 128 dates

    const int n = a.n, Nx = a.Nx, Ny = a.Ny;
    const int nb = (n + 31) >> 5;
    const int npairs = nb * (nb + 1) / 2;
    const size_t CS = 2 * (size_t)n;
    const int npx_zero = a.rows * a.cols;      // index of the all-zero record
    const int R0 = a.row0 + blockIdx.y * a.TH, C0 = blockIdx.x * a.TW;
    const int row_end = a.row0 + a.chunk_rows;
    const int Wx = 2 * Nx + 1, Wn = (2 * Ny + 1) * Wx;
    const int m = lane & 31, half = lane >> 5;

    for (int pid = wave; pid < a.TH * a.TW; pid += WAVES) {
        const int r = R0 + pid / a.TW, c = C0 + pid % a.TW;
        if (r >= row_end || r >= a.rows || c >= a.cols) continue;   // wave-uniform
        const long long pix = (long long)r * a.cols + c;
        const int slot = (r - a.row0) * a.cols + c;
        const uint32_t* w = a.wts + pix * a.nul;
        const bool cen = shp_get(w, shp_flat(0, 0, Nx, Ny));

        // ---- neighbour list ----
        int cnt = 0;
        for (int b0 = 0; b0 < Wn; b0 += 64) {
            const int f = b0 + lane;
            bool take = false;
            int q = 0;
            if (cen && f < Wn) {
                const int rr = r + f / Wx - Ny, cc = c + f % Wx - Nx;
                if (rr >= 0 && rr < a.rows && cc >= 0 && cc < a.cols && shp_get(w, f)) {
                    take = true;
                    q = rr * a.cols + cc;
                }
            }
            const uint64_t bal = __ballot(take);
            if (take) {
                const uint64_t below = (lane == 0) ? 0ull : (bal & ((~0ull) >> (64 - lane)));
                list[cnt + __popcll(below)] = q;
            }
            cnt += __popcll(bal);
        }
        if (!(cen && cnt >= a.min_nb)) {
            if (lane == 0) a.npix[slot] = -1;
            continue;
        }
        const int steps = (cnt + 15) >> 4;
        for (int e = cnt + lane; e < steps * 16; e += 64) list[e] = npx_zero;
        wave_sync_lds();

        float2* gout = (float2*)a.gamma + (size_t)slot * n * n;
        for (int p = 0; p < npairs; ++p) {   // uniform
            int I = p, J = p;
            if (p >= nb) {   // off-diagonal pairs in row order
                int q = p - nb;
                I = 0;
                while (q >= nb - 1 - I) {
                    q -= nb - 1 - I;
                    ++I;
                }
                J = I + 1 + q;
            }
            const int di = 32 * I + m, dj = 32 * J + m;
            const bool vi = di < n, vj = dj < n;
            const int oi = vi ? di : 0, oj = vj ? dj : 0;   // in (re, im) word pairs
            f32x16 RR, II, RI, IR;
#pragma unroll
            for (int v = 0; v < 16; ++v) RR[v] = II[v] = RI[v] = IR[v] = 0.0f;
            for (int s = 0; s < steps; ++s) {
                const int* lp = list + 16 * s + 8 * half;
                uint2 wi[8], wj[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint2* rec = (const uint2*)(a.pk + (size_t)(uint32_t)lp[e] * CS);
                    wi[e] = rec[oi];   // valid address for every lane
                    wj[e] = rec[oj];
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (!vi) wi[e] = make_uint2(0u, 0u);
                    if (!vj) wj[e] = make_uint2(0u, 0u);
                }
                u32x4 rih, ril, iih, iil, rjh, rjl, ijh, ijl;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    rih[e] = __builtin_amdgcn_perm(wi[2 * e + 1].x, wi[2 * e].x, 0x05040100u);
                    ril[e] = __builtin_amdgcn_perm(wi[2 * e + 1].x, wi[2 * e].x, 0x07060302u);
                    iih[e] = __builtin_amdgcn_perm(wi[2 * e + 1].y, wi[2 * e].y, 0x05040100u);
                    iil[e] = __builtin_amdgcn_perm(wi[2 * e + 1].y, wi[2 * e].y, 0x07060302u);
                    rjh[e] = __builtin_amdgcn_perm(wj[2 * e + 1].x, wj[2 * e].x, 0x05040100u);
                    rjl[e] = __builtin_amdgcn_perm(wj[2 * e + 1].x, wj[2 * e].x, 0x07060302u);
                    ijh[e] = __builtin_amdgcn_perm(wj[2 * e + 1].y, wj[2 * e].y, 0x05040100u);
                    ijl[e] = __builtin_amdgcn_perm(wj[2 * e + 1].y, wj[2 * e].y, 0x07060302u);
                }
                const frag_t Rh = __builtin_bit_cast(frag_t, rih), Rl = __builtin_bit_cast(frag_t, ril);
                const frag_t Ih = __builtin_bit_cast(frag_t, iih), Il = __builtin_bit_cast(frag_t, iil);
                const frag_t Sh = __builtin_bit_cast(frag_t, rjh), Sl = __builtin_bit_cast(frag_t, rjl);
                const frag_t Th = __builtin_bit_cast(frag_t, ijh), Tl = __builtin_bit_cast(frag_t, ijl);
                RR = Frag<F16>::mfma(Rh, Sh, RR);
                RR = Frag<F16>::mfma(Rh, Sl, RR);
                RR = Frag<F16>::mfma(Rl, Sh, RR);
                II = Frag<F16>::mfma(Ih, Th, II);
                II = Frag<F16>::mfma(Ih, Tl, II);
                II = Frag<F16>::mfma(Il, Th, II);
                RI = Frag<F16>::mfma(Rh, Th, RI);
                RI = Frag<F16>::mfma(Rh, Tl, RI);
                RI = Frag<F16>::mfma(Rl, Th, RI);
                IR = Frag<F16>::mfma(Ih, Sh, IR);
                IR = Frag<F16>::mfma(Ih, Sl, IR);
                IR = Frag<F16>::mfma(Il, Sh, IR);
            }
            if (I == J) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (acc_row(v, lane) == m) dg[32 * I + m] = RR[v] + II[v];
                wave_sync_lds();
            }
            const int j = 32 * J + m;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int i = 32 * I + acc_row(v, lane);
                if (i >= n || j >= n || i > j) continue;
                float gr = 1.0f, gi = 0.0f;
                if (i != j) {
                    const float sc = rsqrtf(dg[i] * dg[j]);
                    gr = (RR[v] + II[v]) * sc;
                    gi = (IR[v] - RI[v]) * sc;   // P(im_i, re_j) - P(re_i, im_j)
                }
                gout[(size_t)i * n + j] = make_float2(gr, gi);
                if (i != j) gout[(size_t)j * n + i] = make_float2(gr, -gi);
            }
        }
        if (lane == 0) a.npix[slot] = cnt;
        wave_sync_lds();
    }
}

// ---------------------------------------------------------------------------
// Up to 64 dates: the records of the union of a workgroup's windows are staged
// in LDS once, and the waves take their pixels' neighbour lists from there.
// A TH x TW pixel tile needs (TH + 2Ny) x (TW + 2Nx) positions: for 4 x 8
// pixels and a 15 x 11 window that is 308 records for 32 pixels, against
// 165 per pixel gathered one by one.
//
// Dates are padded to NB blocks of 16, products are v_mfma_f32_16x16x32 (32
// positions each; lane l holds date l % 16 and eight positions).  With the
// samples' halves h + l of re (R) and im (I), a diagonal block pair needs
//   A = Rh Rh' + Ih Ih',  X = Rh Rl' + Ih Il',  W = Ih Rh' + Ih Rl' + Il Rh':
//   Re G = A + X + X',  Im G = W - W',
// seven MFMAs instead of the twelve that the four real products take; the
// transposes stay in registers.  A pair I < J takes twelve, into one
// accumulator each for Re G and Im G, and its mirror is its transpose.
//
// Bound by the matrix instructions and the vector unit (operand permutes, list,
// fold) together, and at 30 dates by Gamma's 8 n^2 bytes per pixel (2.8 TB/s).
// Measured against 32 x 32 x 16 products of all four real Grams up to 32 dates
// (2048 x 2048 of 30 dates 14.7 -> 10.9 ms, 640 x 640 of 20 1.40 -> 1.03, 256 x
// 256 of 10 0.18 -> 0.06) and against the gathering kernel above (208 x 224 of
// 48 dates 0.87 -> 0.24 ms, 131 k pixels of 64 dates in a 21 x 11 window 4.5 ->
// 2.3).
// Workgroups are numbered so that each XCD (which owns an L2) takes a
// contiguous run of tiles and the halos neighbouring tiles share stay in it.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <bool F16> __device__ __forceinline__ f32x4 mfma16(typename Frag<F16>::type a, typename Frag<F16>::type b, f32x4 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Transpose of a 16 x 16 accumulator (lane l, register v: row 4 (l / 16) + v,
// column l % 16): the 4 x 4 blocks within each quad of lanes, then the blocks.
template <int CTRL> __device__ __forceinline__ float quad_swap(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ f32x4 transpose16(f32x4 a, int lane) {
    const bool o1 = lane & 1, o2 = lane & 2;
    f32x4 s, c;   // (the swaps by every lane, then the choice)
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] = quad_swap<0xB1>(a[v ^ 1]);
#pragma unroll
    for (int v = 0; v < 4; ++v) a[v] = o1 == ((v & 1) != 0) ? a[v] : s[v];
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] = quad_swap<0x4E>(a[v ^ 2]);
#pragma unroll
    for (int v = 0; v < 4; ++v) c[v] = o2 == ((v & 2) != 0) ? a[v] : s[v];
    const int from = 4 * (4 * (lane >> 4) + (lane & 3) + 4 * (lane & 12));
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float x = c[v];   // (a bit cast of the element itself takes element 0)
        c[v] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(x)));
    }
    return c;
}

// The staged records, padded to 16 NB dates (zeros beyond n and outside the
// image), eight loads of one or two dates in flight.  A group of 16 lanes
// reads half of the 64 banks; with an even NB the date blocks of odd positions
// change places, so that two groups on neighbouring positions read different
// halves.
template <typename V, int NB>
__device__ __forceinline__ void stage_records(const MfmaArgs& a, uint2* rec, int rbase, int cbase, int WC, int NPOS) {
    constexpr int U = sizeof(V) / 8, DP = 16 * NB / U;
    const int n = a.n / U, NT = blockDim.x, total = (NPOS + 1) * DP;
    const V* src = (const V*)a.pk;
    for (int e0 = threadIdx.x; e0 < total; e0 += 8 * NT) {
        V v[8];
        bool in[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = e0 + u * NT;
            const int pos = e / DP, d = e % DP;
            const int rr = rbase + pos / WC, cc = cbase + pos % WC;
            in[u] = e < total && d < n && pos < NPOS && rr >= 0 && rr < a.rows && cc >= 0 && cc < a.cols;
            // slots without data read record 0 and are zeroed below
            const size_t at = in[u] ? ((size_t)rr * a.cols + cc) * n + d : 0;
            v[u] = src[at];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int e = e0 + u * NT;
            const int at = NB % 2 == 0 ? e ^ (((e / DP) & 1) * (16 / U)) : e;
            if (e < total) ((V*)rec)[at] = in[u] ? v[u] : V{};
        }
    }
}

// Waves of the largest tile's workgroup: four and two per SIMD is what the
// registers and LDS allow (two workgroups per CU up to 16 dates).
constexpr int stage_waves(int nb) { return nb == 1 ? 12 : nb == 2 ? 16 : 8; }
template <bool F16, int NB>
__global__ __launch_bounds__(64 * stage_waves(NB)) __attribute__((amdgpu_waves_per_eu(NB <= 2 ? 4 : 2))) void
gram_mfma_lds(MfmaArgs a) {
    const int NT = blockDim.x, WAVES = NT >> 6;
    constexpr int DP = 16 * NB;          // dates of a staged record
    constexpr int PAIRS = NB * (NB - 1) / 2;
    typedef typename Frag<F16>::type frag_t;
    extern __shared__ __align__(16) char smem[];
    const int n = a.n, Nx = a.Nx, Ny = a.Ny;
    const int TH = a.TH, tw = 31 - __builtin_clz(a.TW), TW = 1 << tw;   // TW is a power of two
    const int WR = TH + 2 * Ny, WC = TW + 2 * Nx, NPOS = WR * WC;
    uint2* rec = (uint2*)smem;                             // [NPOS + 1][DP] (re, im) words
    // (the list holds whole addresses: the compiler adds the base to an offset
    // at every load, although it is zero)
    typedef const uint2 __attribute__((address_space(3))) * lds_word;
    const int rec0 = (int)(uintptr_t)(lds_word)rec;
    // wave index in a scalar register, so the pixel loop below is uniform
    // control flow (scalar branches) rather than exec-masked
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int* offs = (int*)(rec + (size_t)(NPOS + 1) * DP);      // window offsets, row << 16 | column
    int* list = offs + a.list_cap + wave * (a.list_cap + DP + kStageWords);
    float* dg = (float*)(list + a.list_cap);                // diagonal of Re G, DP
    uint32_t* wbuf = (uint32_t*)(dg + DP);                  // next pixel's mask words

    // XCD-aware tile order (blocks are dealt to the 8 XCDs round-robin)
    const unsigned nb = gridDim.x * gridDim.y, bid = blockIdx.y * gridDim.x + blockIdx.x;
    const unsigned xcd = bid % 8u, q8 = nb / 8u, rem = nb % 8u;
    const unsigned logical = xcd * q8 + min(xcd, rem) + bid / 8u;
    const int tx = (int)(logical % gridDim.x), ty = (int)(logical / gridDim.x);
    const int R0 = a.row0 + ty * TH, C0 = tx * TW;
    const int row_end = a.row0 + a.chunk_rows;
    const int rbase = R0 - Ny, cbase = C0 - Nx;

    if (n & 1) stage_records<uint2, NB>(a, rec, rbase, cbase, WC, NPOS);
    else stage_records<uint4, NB>(a, rec, rbase, cbase, WC, NPOS);   // records are 16-byte aligned
    const int Wx = 2 * Nx + 1, Wn = (2 * Ny + 1) * Wx;
    for (int f = threadIdx.x; f < Wn; f += NT) offs[f] = f / Wx * 65536 + f % Wx;
    __syncthreads();
    const int m = lane & 15, q = lane >> 4;

    // mask words of a pixel in lanes 0..nul-1 (one load).  The next pixel's
    // are requested at the top of an iteration and parked in LDS before this
    // pixel's Gamma stores, so no wait for them ever waits for the stores.
    auto mask_word = [&](int pid) -> uint32_t {
        const int r = R0 + (pid >> tw), c = C0 + (pid & (TW - 1));
        const bool ok = pid < TH * TW && r < row_end && r < a.rows && c < a.cols;
        // always one load, of pixel 0 when there is no pixel (such a pixel is
        // skipped before its word is used)
        const long long px = ok ? (long long)r * a.cols + c : 0;
        return a.wts[px * a.nul + (lane < a.nul ? lane : 0)];
    };
    if (lane < kStageWords) wbuf[lane] = mask_word(wave);
    for (int pid = wave; pid < TH * TW; pid += WAVES) {
        const uint32_t wword = wbuf[lane & (kStageWords - 1)];
        const uint32_t wnext = mask_word(pid + WAVES);
        const int r = R0 + (pid >> tw), c = C0 + (pid & (TW - 1));
        if (r >= row_end || r >= a.rows || c >= a.cols) {   // wave-uniform
            if (lane < kStageWords) wbuf[lane] = wnext;
            continue;
        }
        const int slot = (r - a.row0) * a.cols + c;
        const int fc = shp_flat(0, 0, Nx, Ny);
        // mask words reach the lanes through readlane (scalar registers), not
        // through an LDS-routed shuffle
        const bool cen = (__builtin_amdgcn_readlane(wword, fc >> 5) >> (fc & 31)) & 1u;
        // ---- neighbour list: LDS addresses of staged records.  Entry k goes
        // to the k % 4'th group of 16 lanes, whose eight entries of a step
        // are contiguous ----
        const int lr = r - R0, lc = c - C0;                  // window origin in the stage
        auto place = [](int k) { return (k & ~31) | ((k & 3) << 3) | ((k >> 2) & 7); };
        auto where = [&](int pos) { return rec0 + (NB % 2 == 0 ? pos * (DP * 8) + ((pos & 1) << 7) : pos * (DP * 8)); };
        int cnt = 0;
        for (int it = 0; it * 64 < Wn; ++it) {
            const int f = it * 64 + lane;
            // lanes 0..31 test word 2it, lanes 32..63 word 2it+1 (lanes past
            // the last word hold word 0 and only cover positions >= Wn)
            const uint32_t wlo = __builtin_amdgcn_readlane(wword, 2 * it);
            const uint32_t whi = __builtin_amdgcn_readlane(wword, 2 * it + 1);
            const uint32_t wf = lane < 32 ? wlo : whi;
            bool take = false;
            int qpos = 0;
            if (cen && f < Wn) {
                const int o = offs[f], fy = o >> 16, fx = o & 0xffff;
                const int rr = r + fy - Ny, cc = c + fx - Nx;
                if (rr >= 0 && rr < a.rows && cc >= 0 && cc < a.cols && ((wf >> (f & 31)) & 1u)) {
                    take = true;
                    qpos = (lr + fy) * WC + (lc + fx);
                }
            }
            const uint64_t bal = __ballot(take);
            if (take) {
                const uint64_t below = (lane == 0) ? 0ull : (bal & ((~0ull) >> (64 - lane)));
                list[place(cnt + __popcll(below))] = where(qpos);
            }
            cnt += __popcll(bal);
        }
        if (!(cen && cnt >= a.min_nb)) {
            if (lane < kStageWords) wbuf[lane] = wnext;
            if (lane == 0) a.npix[slot] = -1;
            continue;
        }
        const int steps = (cnt + 31) >> 5;
        for (int e = cnt + lane; e < steps * 32; e += 64) list[place(e)] = where(NPOS);
        wave_sync_lds();

        // A rounding of a large sum costs more than one of a small: Im Im' has
        // a sum of its own, and so have the halves' cross products (2^-11 of
        // the others) of the pairs.  Where the registers do not hold those,
        // 32 positions are summed by themselves and then added.  (One sum for
        // all: coherence error 1.01 to 1.16 times that of the four real
        // products of 32 x 32 x 16, now 0.88 to 1.01; 160 x 219 pixels of 40
        // dates 200 -> 201 us.)
        constexpr bool OWN = NB <= 3, KEEP = NB == 3;
        f32x4 A[NB], B[NB], X[NB], W[NB], P[PAIRS ? PAIRS : 1], Q[PAIRS ? PAIRS : 1];
        f32x4 PL[KEEP && PAIRS ? PAIRS : 1], QL[KEEP && PAIRS ? PAIRS : 1];
#pragma unroll
        for (int b = 0; b < NB; ++b) A[b] = B[b] = X[b] = W[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < PAIRS; ++t) {
            P[t] = Q[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (KEEP) PL[t] = QL[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        // operands of step st + 1 are loaded while step st's MFMAs run; one
        // 8-byte read gives this lane's (re, im) words of a position
        uint2 x[NB][8];
        auto load_step = [&](int st) {
            const int4* lp = (const int4*)(list + 32 * st + 8 * q);
            const int4 l0 = lp[0], l1 = lp[1];
            const int at[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int o = at[e] + 8 * m;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const lds_word w = (lds_word)(uintptr_t)(uint32_t)(NB % 2 == 0 ? o ^ (b << 7) : o + (b << 7));
                    x[b][e] = make_uint2(w->x, w->y);
                }
            }
        };
        load_step(0);
        for (int st = 0; st < steps; ++st) {
            frag_t Rh[NB], Rl[NB], Ih[NB], Il[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                u32x4 hr, lr4, hi4, li4;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hr[e] = __builtin_amdgcn_perm(x[b][2 * e + 1].x, x[b][2 * e].x, 0x05040100u);
                    lr4[e] = __builtin_amdgcn_perm(x[b][2 * e + 1].x, x[b][2 * e].x, 0x07060302u);
                    hi4[e] = __builtin_amdgcn_perm(x[b][2 * e + 1].y, x[b][2 * e].y, 0x05040100u);
                    li4[e] = __builtin_amdgcn_perm(x[b][2 * e + 1].y, x[b][2 * e].y, 0x07060302u);
                }
                Rh[b] = __builtin_bit_cast(frag_t, hr);
                Rl[b] = __builtin_bit_cast(frag_t, lr4);
                Ih[b] = __builtin_bit_cast(frag_t, hi4);
                Il[b] = __builtin_bit_cast(frag_t, li4);
            }
            load_step(st + 1 < steps ? st + 1 : st);
            // interleaved so that consecutive MFMAs feed different accumulators
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                B[b] = OWN ? B[b] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                (OWN ? A[b] : B[b]) = mfma16<F16>(Rh[b], Rh[b], OWN ? A[b] : B[b]);
                X[b] = mfma16<F16>(Rh[b], Rl[b], X[b]);
                W[b] = mfma16<F16>(Ih[b], Rh[b], W[b]);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                B[b] = mfma16<F16>(Ih[b], Ih[b], B[b]);
                X[b] = mfma16<F16>(Ih[b], Il[b], X[b]);
                W[b] = mfma16<F16>(Ih[b], Rl[b], W[b]);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                W[b] = mfma16<F16>(Il[b], Rh[b], W[b]);
                if constexpr (!OWN) A[b] += B[b];
            }
            int t = 0;
#pragma unroll
            for (int b = 0; b < NB - 1; ++b) {
                const u32x4 sign = {0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
                const frag_t Nh = __builtin_bit_cast(frag_t, __builtin_bit_cast(u32x4, Rh[b]) ^ sign);
                const frag_t Nl = __builtin_bit_cast(frag_t, __builtin_bit_cast(u32x4, Rl[b]) ^ sign);
#pragma unroll
                for (int d = b + 1; d < NB; ++d, ++t) {   // P(im_b, re_d) - P(re_b, im_d) is Im G
                    f32x4 p = f32x4{0.0f, 0.0f, 0.0f, 0.0f}, q = p, pl = p, ql = p;
                    if constexpr (KEEP) p = P[t], q = Q[t], pl = PL[t], ql = QL[t];
                    p = mfma16<F16>(Rh[b], Rh[d], p);
                    q = mfma16<F16>(Ih[b], Rh[d], q);
                    pl = mfma16<F16>(Rh[b], Rl[d], pl);
                    ql = mfma16<F16>(Ih[b], Rl[d], ql);
                    p = mfma16<F16>(Ih[b], Ih[d], p);
                    q = mfma16<F16>(Nh, Ih[d], q);
                    pl = mfma16<F16>(Rl[b], Rh[d], pl);
                    ql = mfma16<F16>(Il[b], Rh[d], ql);
                    pl = mfma16<F16>(Ih[b], Il[d], pl);
                    ql = mfma16<F16>(Nh, Il[d], ql);
                    pl = mfma16<F16>(Il[b], Ih[d], pl);
                    ql = mfma16<F16>(Nl, Ih[d], ql);
                    if constexpr (KEEP) {
                        P[t] = p;
                        Q[t] = q;
                        PL[t] = pl;
                        QL[t] = ql;
                    } else {
                        P[t] += p + pl;
                        Q[t] += q + ql;
                    }
                }
            }
        }

        if (lane < kStageWords) wbuf[lane] = wnext;   // waits for the load here, before the stores below

        // ---- fold into Gamma ----
        if constexpr (OWN) {
#pragma unroll
            for (int b = 0; b < NB; ++b) A[b] += B[b];
        }
        // Re G_mm sits in register m % 4 of the lanes of quarter m / 4; it is
        // published as 1 / sqrt: one transcendental per lane, and the
        // normalisation of entry (i, j) is a product
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float dv = 0.0f;
#pragma unroll
            for (int v = 0; v < 4; ++v) dv = (m & 3) == v ? A[b][v] + (X[b][v] + X[b][v]) : dv;
            if (q == m >> 2) dg[16 * b + m] = rsqrtf(dv);
        }
        wave_sync_lds();
        float2* gout = reinterpret_cast<float2*>(a.gamma) + (size_t)slot * n * n;
        // entries (16 I + 4 q + v, 16 J + m)
        auto put = [&](int I, int J, const f32x4& re, const f32x4& im) {
            const float dj = dg[16 * J + m];
            const int col = 16 * J + m;
            float di[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) di[v] = dg[16 * I + 4 * q + v];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * I + 4 * q + v;
                const float sc = di[v] * dj;
                const bool off = I != J || 4 * q + v != m;
                const float gr = off ? re[v] * sc : 1.0f;
                const float gi = off ? im[v] * sc : 0.0f;
                if (row < n && col < n) gout[(size_t)row * n + col] = make_float2(gr, gi);
            }
        };
        int t = 0;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            put(b, b, A[b] + (X[b] + transpose16(X[b], lane)), W[b] - transpose16(W[b], lane));
#pragma unroll
            for (int d = b + 1; d < NB; ++d, ++t) {
                if constexpr (KEEP) {
                    P[t] += PL[t];
                    Q[t] += QL[t];
                }
                put(b, d, P[t], Q[t]);
                put(d, b, transpose16(P[t], lane), -transpose16(Q[t], lane));
            }
        }
        if (lane == 0) a.npix[slot] = cnt;
        wave_sync_lds();
    }
}

static int gram_list_cap(int Nx, int Ny) {
    const int Wn = (2 * Ny + 1) * (2 * Nx + 1);
    return ((Wn + 15) / 16) * 16 + 16;
}

struct StageTile {
    int TH, TW, waves;
};
// Largest first.  8 x 16 pixels stage ~4.2 records per pixel at a 15 x 11
// window, 4 x 16 ~6.6, 4 x 8 9.7, 2 x 4 27.
constexpr StageTile kStageTiles[] = {{8, 16, 16}, {4, 16, 8}, {4, 8, 8}, {4, 4, 8}, {2, 4, 8}, {2, 2, 4}};

static size_t gram_lds_bytes(int n, int Nx, int Ny, const StageTile& t) {
    const int dp = (n + 15) / 16 * 16;
    const size_t stage = (size_t)((t.TH + 2 * Ny) * (t.TW + 2 * Nx) + 1) * dp * 8;
    const int cap = gram_list_cap(Nx, Ny);   // of the window offsets, too
    return stage + (size_t)cap * 4 + (size_t)t.waves * (cap + dp + kStageWords) * 4;
}

// Tile of the staged kernel: the one with the least estimated time on the
// launch's pixels, in units of a CU's time for a pixel when its waves fill it
// (0.6 us at 30 dates).  A workgroup costs its pixels, and for staging four and
// a hundredth of its positions; those of a CU share it, and a wave's pixels,
// one after the other, take twelve each at least; the launch takes as many
// rounds as it fills the chip.  (64 x 64 pixels of 8
// dates: 32 tiles of 8 x 16 took 77 us, 512 of 2 x 4 take 12; 160 x 219 of 40:
// 560 tiles of 4 x 16 in three rounds 219 us, 2200 of 4 x 4 in nine 198.)  The
// four constants are fitted to the measured times of about twenty sizes, not
// derived.  Where they lead, over 6, 12, 16, 24 and 30 dates, windows of 5 x 5
// to 21 x 11 and 48 x 48 to 1024 x 1024 pixels (120 in all): the median is
// 0.4 % over the best of this choice, 4 x 16 at most and 4 x 8 at most; the
// worst 17 %, at a 21 x 11 window up to 16 dates, where 4 x 16 is faster (1024
// x 1024 of 6: 1.22 and 1.04 ms); next 11 %, 131 x 300 of 12 (41 and 37 us).
// A scheduled variant (FRINGE_GRAM_STAGED12 / 8 / 4) names the largest tile
// tried; one that does not fit the window falls back to the others.  False
// above 64 dates, for windows of more than kStageWords mask words and where
// nothing fits: the gathering kernels walk any number of words.
static bool gram_staged(int n, int Nx, int Ny, long long rows, int cols, StageTile& best, size_t& bytes) {
    if (n > 64 || shp_words(Nx, Ny) > kStageWords) return false;
    const int v = n <= 32 ? schedule_lookup(FRINGE_SCHED_GRAM_VARIANT, n, Nx, Ny, FRINGE_GRAM_DEFAULT) : FRINGE_GRAM_DEFAULT;
    if (v == FRINGE_GRAM_UNSTAGED) return false;
    const int from = v == FRINGE_GRAM_STAGED8 ? 1 : v == FRINGE_GRAM_STAGED4 ? 2 : 0;
    const int blocks = (n + 15) / 16, most = blocks == 1 ? 28 : blocks == 2 ? 16 : 8;   // waves of a CU, by registers
    bool found = false;
    double least = 0.0;
    for (int k = from; k < (int)(sizeof(kStageTiles) / sizeof(kStageTiles[0])); ++k) {
        StageTile t = kStageTiles[k];
        t.waves = std::min(t.waves, stage_waves(blocks));
        const size_t b = gram_lds_bytes(n, Nx, Ny, t);
        if (b > 160 * 1024) continue;
        if ((long long)((cols + t.TW - 1) / t.TW) * 64 * t.waves >= 1ll << 32) continue;   // threads of a launch's x
        const long long wgs = (long long)((cols + t.TW - 1) / t.TW) * ((rows + t.TH - 1) / t.TH);
        const int fit = (int)std::min<size_t>(160 * 1024 / b, (size_t)std::max(most / t.waves, 1));
        const int active = (int)std::min<long long>(fit, (wgs + 255) / 256), px = t.TH * t.TW;
        const double stage = 4 + 0.01 * (t.TH + 2 * Ny) * (t.TW + 2 * Nx);
        const double cost = (double)((wgs + 256ll * active - 1) / (256ll * active)) *
                            std::max(active * (px + stage), 12.0 * ((px + t.waves - 1) / t.waves) + stage);
        if (found && cost >= least) continue;
        best = t;
        bytes = b;
        least = cost;
        found = true;
    }
    return found;
}

int gram_stage_rows(int n, int Nx, int Ny) {
    StageTile t;
    size_t bytes;
    return n <= 32 && gram_staged(n, Nx, Ny, 1ll << 30, 1 << 20, t, bytes) ? t.TH : 1;
}

// packed records followed by the per-date maxima (256-byte aligned)
size_t mfma_pack_bytes(int rows, int cols, int n) {
    const size_t rec = ((size_t)rows * cols + 1) * 2 * n * sizeof(uint32_t);
    return ((rec + 255) & ~(size_t)255) + (size_t)n * sizeof(uint32_t);
}

int pack_launch(const float2* slc, int rows, int cols, int n, bool f16, uint32_t* pk, int* count, hipStream_t s) {
    const long long npx = (long long)rows * cols;
    const size_t rec = ((size_t)npx + 1) * 2 * n * sizeof(uint32_t);
    uint32_t* dmax = (uint32_t*)((char*)pk + ((rec + 255) & ~(size_t)255));
    const unsigned blocks = (unsigned)((npx + 63) / 64);
    if (f16) {
        // one workgroup per date needs no cleared words, and a launch less
        // outweighs its fewer loads in flight: calls back to back of 64 x 64
        // pixels of 8 dates 38 -> 31 us, 128 x 128 of 30 212 -> 197, 140 x 140
        // of 8 87.6 -> 83.2; at 256 x 256 (of 10, 209.5 and 208.2) the two are
        // level, so the line lies there
        if (npx <= 65536) {
            hipLaunchKernelGGL(date_absmax<1024>, dim3(1, n), dim3(1024), 0, s, slc, npx, dmax);
        } else {
            hipLaunchKernelGGL(date_absmax_clear, dim3((n + 63) / 64), dim3(64), 0, s, dmax, n);
            // 64 workgroups per date
            hipLaunchKernelGGL(date_absmax<256>, dim3(64, n), dim3(256), 0, s, slc, npx, dmax);
        }
        hipLaunchKernelGGL(pack_hilo<true>, dim3(blocks), dim3(256), (size_t)64 * 2 * n * 4, s, slc, n,
                           npx, (const uint32_t*)dmax, pk, count);
    } else {
        hipLaunchKernelGGL(pack_hilo<false>, dim3(blocks), dim3(256), (size_t)64 * 2 * n * 4, s, slc, n,
                           npx, (const uint32_t*)dmax, pk, count);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int NBH, int WAVES, bool F16>
static void launch_mfma(MfmaArgs a, hipStream_t s) {
    const size_t wbytes = (size_t)a.list_cap * 4 + 32 * 33 * 4 + 64 * NBH * 4;
    const dim3 grid((unsigned)((a.cols + a.TW - 1) / a.TW),
                    (unsigned)((a.chunk_rows + a.TH - 1) / a.TH));
    hipLaunchKernelGGL((gram_mfma<NBH, WAVES, F16>), grid, dim3(64 * WAVES), wbytes * WAVES, s, a);
}

template <bool F16> static void launch_staged(const MfmaArgs& a, int waves, size_t bytes, hipStream_t s) {
    const dim3 grid((unsigned)((a.cols + a.TW - 1) / a.TW), (unsigned)((a.chunk_rows + a.TH - 1) / a.TH));
    const dim3 blk(64 * waves);
    switch ((a.n + 15) / 16) {   // blocks of 16 dates
        case 1: hipLaunchKernelGGL((gram_mfma_lds<F16, 1>), grid, blk, bytes, s, a); break;
        case 2: hipLaunchKernelGGL((gram_mfma_lds<F16, 2>), grid, blk, bytes, s, a); break;
        case 3: hipLaunchKernelGGL((gram_mfma_lds<F16, 3>), grid, blk, bytes, s, a); break;
        default: hipLaunchKernelGGL((gram_mfma_lds<F16, 4>), grid, blk, bytes, s, a); break;
    }
}

int gram_mfma_launch(const LinkPlan& P, const uint32_t* pk, const uint32_t* wts, long long first,
                     int slots, hipStream_t s) {
    if (P.n > kMaxBandsMfma || first % P.cols != 0 || slots % P.cols != 0) return -1;
    MfmaArgs a{};
    a.pk = pk;
    a.wts = wts;
    a.rows = P.rows;
    a.cols = P.cols;
    a.n = P.n;
    a.Nx = P.Nx;
    a.Ny = P.Ny;
    a.nul = P.nul;
    a.min_nb = P.min_nb;
    a.row0 = (int)(first / P.cols);
    a.chunk_rows = slots / P.cols;
    a.TH = 2;
    a.TW = 8;
    a.gamma = (float*)P.d_gamma;
    a.npix = P.d_npix;
    a.list_cap = gram_list_cap(P.Nx, P.Ny);
    const bool f16 = (P.precision != FRINGE_PREC_MIXED_BF16);
    StageTile t;
    size_t bytes = 0;
    if (gram_staged(P.n, P.Nx, P.Ny, a.chunk_rows, P.cols, t, bytes)) {
        a.TH = t.TH;
        a.TW = t.TW;
        if (f16) launch_staged<true>(a, t.waves, bytes, s);
        else launch_staged<false>(a, t.waves, bytes, s);
    } else if (P.n <= 32) {
        if (f16) launch_mfma<1, 4, true>(a, s);
        else launch_mfma<1, 4, false>(a, s);
    } else {
        const size_t wbytes = (size_t)a.list_cap * 4 + 128 * 4;
        const dim3 grid((unsigned)((a.cols + a.TW - 1) / a.TW), (unsigned)((a.chunk_rows + a.TH - 1) / a.TH));
        if (f16) hipLaunchKernelGGL((gram_mfma_pairs<4, true>), grid, dim3(256), wbytes * 4, s, a);
        else hipLaunchKernelGGL((gram_mfma_pairs<4, false>), grid, dim3(256), wbytes * 4, s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace fringe
