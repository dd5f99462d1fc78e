// bf_dftmm.h -- line transforms of any length n < 1024 that is no power of two
// >= 16 (the reference's 101^2 grid among them) as products with a cosine and a
// sine matrix on the FP64 matrix cores.
//
// With H = n/2 (floor), e_0 = x_0, e_j = x_j + x_{n-j}, o_j = x_j - x_{n-j}
// (1 <= j, 2j < n) and e_{n/2} = x_{n/2} for even n,
//     X_k     = sum_j e_j cos(2 pi j k / n) - i sum_j o_j sin(2 pi j k / n)
//     X_{n-k} = sum_j e_j cos(2 pi j k / n) + i sum_j o_j sin(2 pi j k / n),
// k = 0..H: two real matrices of a quarter of the DFT matrix's entries applied to
// complex data, 2 n^2 flop per line against 8 n^2 for the direct sum.  The inverse
// (unnormalised, as fft/ifft share the factor with the phase table) takes +i.
// Inputs known to be zero outside a band of lines and outputs needed only inside
// it shorten the contraction and the output range: the aperture's band
// [lo, hi) becomes the range [min(lo, n - hi + 1), H] of the folded index j.
//
// A block holds 8 complex lines.  Their folded values sit in LDS as two planes
// (e and -+i o) of rows [j][16]: columns 0..7 the real parts, 8..15 the imaginary
// parts of the 8 lines.  v_mfma_f64_16x16x4f64 takes the planes as A (row i =
// line/part) and the matrix as B (column = output index), so a lane of the result
// holds both parts of two lines (lane/16 and 4 + lane/16) at one output index
// and, as E + O and E - O, at its mirror: the k-space phase, the boundary update,
// the aperture mask and the next fold all stay in the lane.  A wave owns an
// output tile of 16; where an output range has fewer tiles than the block has
// waves, two or four waves share the contraction and add their partial tiles through LDS.
#pragma once
#include "bf_device.h"

namespace bf {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// plane row stride in doubles: the mid-stage writes (16 consecutive rows per
// quarter wave) spread over the banks, the reads stay 16 consecutive doubles
constexpr int DFT_LDP = 18;
constexpr int DFT_LINES = 8;
constexpr int DFT_PART = 512;  // doubles of one wave's partial tile pair

__host__ __device__ inline int dft_rows(int n, int a0) { return ((n / 2 - a0 + 1) + 3) & ~3; }
__host__ __device__ inline int dft_tiles(int n, int b0) { return (n / 2 - b0 + 16) / 16; }
// row stride of the cosine/sine matrix: contraction rows reach H + 3, output tiles H + 15
__host__ __device__ inline int dft_ld(int n) { return (n / 2 + 17 + 15) & ~15; }
// smallest folded index of the lines [lo, hi) (0 when the range is empty or everything)
__host__ __device__ inline int dft_fold_lo(int n, int lo, int hi) {
    if (hi <= lo) return 0;
    const int m = lo < n - hi + 1 ? lo : n - hi + 1;
    return m < 0 ? 0 : m > n / 2 ? n / 2 : m;
}
// the index has a mirror of its own
__device__ __forceinline__ bool dft_paired(int n, int j) { return j > 0 && 2 * j < n; }

// folds (x, mirror) into plane row `row`, line `c`; INV: +i o, else -i o
template <bool INV>
__device__ __forceinline__ void dft_fold(double* E, double* O, int row, int c, bool paired, zd x, zd m) {
    double* e = E + row * DFT_LDP + c;
    double* o = O + row * DFT_LDP + c;
    if (paired) {
        e[0] = x.re + m.re;
        e[8] = x.im + m.im;
        const double dr = x.re - m.re, di = x.im - m.im;
        o[0] = INV ? -di : di;
        o[8] = INV ? dr : -dr;
    } else {
        e[0] = x.re;
        e[8] = x.im;
        o[0] = 0.0;
        o[8] = 0.0;
    }
}

// One transform stage: contraction over the folded indices a0 .. H (a0 a multiple
// of 4; plane row 0 is a0), outputs b0 + 16 tile + lane%16 for mt tiles.  Returns
// whether this wave owns the tiles tile0, tile0 + waves, ... (those < mt).  A
// barrier before the first plane read and one after the last: the planes the block
// has just written are read, and may be overwritten afterwards.
// The contraction is cut into the four quarters of the whole range 0 .. H, added as
// (c0 + c1) + (c2 + c3): smax = 4 lets two or four waves share a tile (part holds
// their partial tiles), and the result's bits depend neither on that nor on a0.
template <int TPW>
__device__ __forceinline__ bool dft_stage(const double* E, const double* O, double* part, int n, int a0, int b0,
                                          int mt, int smax, const double2* __restrict__ T, int ld, dbl4 (&e)[TPW],
                                          dbl4 (&o)[TPW], int& tile0) {
    const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int i = lane & 15, kk = lane >> 4;
    const int KF = dft_rows(n, 0) >> 2, ka = a0 >> 2;  // steps of 4: the whole range, the first one needed
    const int S = smax >= 4 && W >= 4 * mt ? 4 : smax >= 4 && W >= 2 * mt ? 2 : 1;
    const int first = wave / S, s = wave - first * S;
    const int c0 = s * (4 / S), c1 = c0 + 4 / S;
    const int kb = KF * c0 / 4, kbeg = kb > ka ? kb : ka;
    const double2* t = T + (size_t)kk * ld + b0 + 16 * first + i;
    const size_t step = 4 * (size_t)ld;
    // matrix entries a group of four steps ahead of their products (the first ones before the barrier)
    double2 w[4];
    auto fetch = [&](int k) {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = t[step * (k + u < KF ? k + u : KF - 1)];
    };
    if (first < mt)
        fetch(kbeg);
    else
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = make_double2(0, 0);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        e[q] = dbl4{0, 0, 0, 0};
        o[q] = dbl4{0, 0, 0, 0};
        const int tile = first + q * W;
        if (tile < mt && (q == 0 || S == 1)) {
            if (q > 0) {
                t += 16 * W;
                fetch(kbeg);
            }
            int k = kbeg;
            dbl4 pe{0, 0, 0, 0}, po{0, 0, 0, 0};
            for (int c = c0; c < c1; c++) {
                const int hi = KF * (c + 1) / 4;
                dbl4 ce{0, 0, 0, 0}, co{0, 0, 0, 0};
                while (k < hi) {
                    const int nk = k + 4 < hi ? k + 4 : hi;
                    double2 v[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) v[u] = w[u];
                    fetch(nk);
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (k + u < nk) {
                            const int p = (4 * (k + u - ka) + kk) * DFT_LDP + i;
                            ce = __builtin_amdgcn_mfma_f64_16x16x4f64(E[p], v[u].x, ce, 0, 0, 0);
                            co = __builtin_amdgcn_mfma_f64_16x16x4f64(O[p], v[u].y, co, 0, 0, 0);
                        }
                    k = nk;
                }
                if (c & 1) {  // the pair's second quarter
                    e[q] += pe + ce;
                    o[q] += po + co;
                    pe = dbl4{0, 0, 0, 0};
                    po = dbl4{0, 0, 0, 0};
                } else {
                    pe = ce;
                    po = co;
                }
            }
            if (S == 4 && !(c0 & 1)) {
                e[q] = pe;
                o[q] = po;
            }
        }
    }
    tile0 = first;
    const bool own = first < mt && s == 0;
    if (S > 1) {
        double* pt = part + (size_t)(first * (S - 1)) * DFT_PART + lane;
        if (first < mt && s > 0) {
            double* w = pt + (s - 1) * DFT_PART;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                w[v * 64] = e[0][v];
                w[(4 + v) * 64] = o[0][v];
            }
        }
        __syncthreads();
        if (own)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                e[0][v] += pt[v * 64];
                o[0][v] += pt[(4 + v) * 64];
                if (S == 4) {
                    e[0][v] += pt[DFT_PART + v * 64] + pt[2 * DFT_PART + v * 64];
                    o[0][v] += pt[DFT_PART + (4 + v) * 64] + pt[2 * DFT_PART + (4 + v) * 64];
                }
            }
    } else {
        __syncthreads();
    }
    return own;
}
// the two lines of a lane (h = 0: line lane/16, h = 1: line 4 + lane/16) at the output index and at its mirror
__device__ __forceinline__ zd dft_out(const dbl4& e, const dbl4& o, int h) {
    return cmk<double>(e[h] + o[h], e[2 + h] + o[2 + h]);
}
__device__ __forceinline__ zd dft_mirror(const dbl4& e, const dbl4& o, int h) {
    return cmk<double>(e[h] - o[h], e[2 + h] - o[2 + h]);
}
// zero plane rows [from, to): the padding of the next contraction
__device__ __forceinline__ void dft_zero_rows(double* E, double* O, int from, int to) {
    for (int q = threadIdx.x; q < (to - from) * 16; q += blockDim.x) {
        const int p = (from + (q >> 4)) * DFT_LDP + (q & 15);
        E[p] = 0.0;
        O[p] = 0.0;
    }
}

}  // namespace bf
