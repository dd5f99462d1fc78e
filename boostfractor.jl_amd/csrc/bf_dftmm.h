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
// A block holds 8 complex lines.  Their folded values sit in LDS as rows [j][16] of
// (e, -+i o) pairs: columns 0..7 the real parts, 8..15 the imaginary parts of the
// 8 lines.  v_mfma_f64_16x16x4f64 takes the rows as A (row i = line/part) and the
// matrix as B (column = output index), so a lane of the result holds both parts of
// two lines (lane/16 and 4 + lane/16) at one output index and, as E + O and E - O,
// at its mirror: the k-space phase, the boundary update, the aperture mask and the
// next fold all stay in the lane.  Indices 0 and n/2, their own mirrors, are folded
// with a zero mirror: their sines are exact zeros.  A wave owns an output tile of
// 16; where an output range has fewer tiles than the block has waves, two or four
// waves share the contraction and add their partial tiles through LDS.
#pragma once
#include "bf_device.h"

namespace bf {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// row stride in pairs: the folds after a transform write 16 consecutive rows per
// quarter wave, which an odd stride spreads over all banks
constexpr int DFT_LDP = 17;
constexpr int DFT_LINES = 8;
constexpr int DFT_PART = 128;  // pairs of one wave's partial tile

__host__ __device__ inline int dft_rows(int n, int a0) { return ((n / 2 - a0 + 1) + 3) & ~3; }
__host__ __device__ inline int dft_tiles(int n, int b0) { return (n / 2 - b0 + 16) / 16; }
// row stride of the cosine/sine matrix: contraction rows reach H + 3, output tiles H + 15
__host__ __device__ inline int dft_ld(int n) { return (n / 2 + 17 + 15) & ~15; }
// rows of the matrix: the loads ahead of the last products reach past H + 3
__host__ __device__ inline int dft_tab_rows(int n) { return dft_ld(n) + 32; }
// smallest folded index of the lines [lo, hi) (0 when the range is empty or everything)
__host__ __device__ inline int dft_fold_lo(int n, int lo, int hi) {
    if (hi <= lo) return 0;
    const int m = lo < n - hi + 1 ? lo : n - hi + 1;
    return m < 0 ? 0 : m > n / 2 ? n / 2 : m;
}
// the index has a mirror of its own
__device__ __forceinline__ bool dft_paired(int n, int j) { return j > 0 && 2 * j < n; }

// folds (x, mirror) into row `row`, line `c`; INV: +i o, else -i o
template <bool INV>
__device__ __forceinline__ void dft_fold(double2* P, int row, int c, zd x, zd m) {
    double2* p = P + row * DFT_LDP + c;
    const double dr = x.re - m.re, di = x.im - m.im;
    p[0] = make_double2(x.re + m.re, INV ? -di : di);
    p[8] = make_double2(x.im + m.im, INV ? dr : -dr);
}
__device__ __forceinline__ double2 dft_entry(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0);
    return make_double2(__hiloint2double((int)v[1], (int)v[0]), __hiloint2double((int)v[3], (int)v[2]));
}

// How the waves of a block share mt output tiles: S waves per tile, this wave's part
// s of tile `first` (and of first + waves, ... when S = 1).  Two waves of a tile take
// its cosine and its sine product, four also halve the contraction.
struct DftShare {
    int S, first, s;
    __device__ __forceinline__ DftShare(int mt, int smax) {
        const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        S = smax >= 4 && W >= 4 * mt ? 4 : smax >= 2 && W >= 2 * mt ? 2 : 1;
        first = wave / S;
        s = wave - first * S;
    }
    __device__ __forceinline__ bool own(int mt) const { return s == 0 && first < mt; }
};

// The contraction steps [k0, k1) of one half of the range, MODE 1: cosines, 2: sines,
// 3: both.  w holds the matrix entries of steps k0 .. k0 + 3 and is left with those of
// the four steps from k1 on.
template <int MODE, typename F>
__device__ __forceinline__ void dft_steps(const double2* pl, int k0, int k1, double2 (&w)[4], F fetch, dbl4& ce,
                                          dbl4& co) {
    for (int k = k0; k < k1;) {
        const int nk = k + 4 < k1 ? k + 4 : k1;
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = w[u];
        fetch(nk);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (k + u < nk) {
                const double2 p = pl[4 * (k + u) * DFT_LDP];
                if constexpr (MODE & 1) ce = __builtin_amdgcn_mfma_f64_16x16x4f64(p.x, v[u].x, ce, 0, 0, 0);
                if constexpr (MODE & 2) co = __builtin_amdgcn_mfma_f64_16x16x4f64(p.y, v[u].y, co, 0, 0, 0);
            }
        k = nk;
    }
}

// One transform stage: contraction over the folded indices a0 .. H (a0 a multiple
// of 4; row 0 of P is a0), outputs b0 + 16 tile + lane%16 for mt tiles, tile =
// sh.first + q waves in e[q], o[q] of the waves that own one (sh.own).  A barrier
// before the first read of P and one after the last: the rows the block has just
// written are read, and may be overwritten afterwards.  The two halves of the whole
// range 0 .. H are summed apart and added, so the result's bits depend neither on
// the waves that share a tile (part holds their partial tiles) nor on a0.
template <int TPW>
__device__ __forceinline__ void dft_stage(const double2* P, double2* part, int n, int a0, int b0, int mt,
                                          const DftShare& sh, const double2* __restrict__ T, dbl4 (&e)[TPW],
                                          dbl4 (&o)[TPW]) {
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int i = lane & 15, kk = lane >> 4;
    const int KF = dft_rows(n, 0) >> 2, KH = KF >> 1, ka = a0 >> 2;  // steps of 4: all, the first half's, the first needed
    const int S = sh.S, first = sh.first, s = sh.s;
    // this wave's halves: [kb, km) and [km, ke)
    const int kb = S == 4 && s >= 2 ? (ka > KH ? ka : KH) : ka;
    const int km = kb > KH ? kb : KH, ke = S == 4 && s < 2 ? km : KF;
    // matrix entries a group of four steps ahead of their products (the first ones before the
    // barrier; the last ones, past H + 3, are not used)
    const int ld = dft_ld(n);
    const auto rt = buf_rsrc(T, (uint32_t)(ld * dft_tab_rows(n)) * (uint32_t)sizeof(double2));
    uint32_t lane0 = (uint32_t)(kk * ld + b0 + 16 * first + i) * (uint32_t)sizeof(double2);
    const uint32_t step = 4 * (uint32_t)ld * (uint32_t)sizeof(double2);
    const double2* pl = P + (kk - 4 * ka) * DFT_LDP + i;
    double2 w[4];
    auto fetch = [&](int k) {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = dft_entry(rt, lane0, step * (uint32_t)(k + u));
    };
    fetch(kb);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        dbl4 e0{0, 0, 0, 0}, o0{0, 0, 0, 0}, e1{0, 0, 0, 0}, o1{0, 0, 0, 0};
        if (first + q * W < mt && (q == 0 || S == 1)) {
            if (q > 0) {
                lane0 += 16 * (uint32_t)W * (uint32_t)sizeof(double2);
                fetch(kb);
            }
            if (S == 1) {
                dft_steps<3>(pl, kb, km, w, fetch, e0, o0);
                dft_steps<3>(pl, km, ke, w, fetch, e1, o1);
            } else if (s & 1) {
                dft_steps<2>(pl, kb, km, w, fetch, e0, o0);
                dft_steps<2>(pl, km, ke, w, fetch, e1, o1);
            } else {
                dft_steps<1>(pl, kb, km, w, fetch, e0, o0);
                dft_steps<1>(pl, km, ke, w, fetch, e1, o1);
            }
        }
        e[q] = e0 + e1;
        o[q] = o0 + o1;
    }
    if (S > 1) {
        // partial tiles of a tile's waves 1 .. S-1, two doubles of a lane side by side
        double2* pt = part + (size_t)(first * (S - 1)) * DFT_PART + lane;
        if (first < mt && s > 0) {
            const dbl4 v = (s & 1) ? o[0] : e[0];
            double2* d = pt + (s - 1) * DFT_PART;
            d[0] = make_double2(v[0], v[1]);
            d[64] = make_double2(v[2], v[3]);
        }
        __syncthreads();
        if (sh.own(mt)) {
            auto get = [&](int r) {
                const double2 x = pt[r * DFT_PART], y = pt[r * DFT_PART + 64];
                return dbl4{x.x, x.y, y.x, y.y};
            };
            o[0] = get(0);
            if (S == 4) {
                e[0] += get(1);
                o[0] += get(2);
            }
        }
    } else {
        __syncthreads();
    }
}
// the two lines of a lane (h = 0: line lane/16, h = 1: line 4 + lane/16) at the output index and at its mirror
__device__ __forceinline__ zd dft_out(const dbl4& e, const dbl4& o, int h) {
    return cmk<double>(e[h] + o[h], e[2 + h] + o[2 + h]);
}
__device__ __forceinline__ zd dft_mirror(const dbl4& e, const dbl4& o, int h) {
    return cmk<double>(e[h] - o[h], e[2 + h] - o[2 + h]);
}
// zero rows [from, to): what the next contraction meets outside the folded values
__device__ __forceinline__ void dft_zero_rows(double2* P, int from, int to) {
    for (int q = threadIdx.x; q < (to - from) * 16; q += blockDim.x)
        P[(from + (q >> 4)) * DFT_LDP + (q & 15)] = make_double2(0, 0);
}

}  // namespace bf
