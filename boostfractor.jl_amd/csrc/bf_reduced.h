// bf_reduced.h -- the bounce solvers' propagation on the aperture's window.
//
// Every propagation of a bounce starts by zeroing the field outside the aperture
// (src/boost_fractor.jl:159), and whatever it leaves outside is zeroed again before
// the next one.  Between two masks the operator is a circular convolution: the field
// on the window of by x bx samples that holds the aperture goes to the same window
// through the kernel h = IFFT(exp(-i kz dz)) at the offsets |dy| < by, |dx| < bx.  A
// circular convolution on My x Mx >= (2 by - 1) x (2 bx - 1) samples, with h cut to
// those offsets, gives the same numbers: on the 1 m grids (0.3 of a side inside the
// aperture) 160^2 instead of 256^2 and 320^2 instead of 512^2 points, a third of the
// lines' arithmetic and 0.6 of the bytes.  The phase tables are replaced by
// DFT_M(cut(IFFT_N(table))), formed in FP64 once per frequency batch.
//
// The outputs on the whole grid are sums over the bounces of propagated fields, so
// the masked fields are summed first (FP64, on the window, transformed along x) and
// the sum is propagated once on the whole grid.
//
// The k range of an even grid is symmetric about half a bin, k = (m + 1/2) dk (about a bin
// for an odd one), so h(d) = exp(-i pi d / N) g(d) with an even g: fields carried with the
// factor exp(i pi y / N) (which commutes with masks, surfaces and boundaries) see the even
// kernel g, whose tables are mirror symmetric and stored as quarters.
//
// Lines have M = 16 R points.  Thread t of 16 holds the samples t + 16 m (m < R, of
// which at most half lie in the window), thread k1 of R the wavenumbers k1 + R k2
// (k2 < 16): one exchange through LDS per transform, radix R on one side and radix 16
// on the other (bf_fftmix.h).
#pragma once
#include "bf_passes.h"

namespace bf {

struct RdShape {
    int Ry = 0, Rx = 0;            // radices: lines of 16 Ry (columns) and 16 Rx (rows) points
    int y0 = 0, by = 0, x0 = 0, bx = 0;  // window in the grid
    double ey = 0, ex = 0;         // phase per sample in units of pi: 1/ny, 1/nx on even grids, else 0
    bool quarter = false;          // mirror-symmetric k range: quarter tables
    int My() const { return 16 * Ry; }
    int Mx() const { return 16 * Rx; }
    size_t field() const { return (size_t)by * Mx(); }  // elements of a stored field: window rows, wavenumbers along x
    size_t points() const { return (size_t)My() * Mx(); }
    size_t table() const { return quarter ? (size_t)(My() / 2 + 1) * (Mx() / 2 + 1) : points(); }
};
// smallest radix whose lines hold the window's convolution, or 0
inline int rd_radix(int b) {
    for (int R : {4, 5, 6, 8, 10, 12, 16, 20})
        if (2 * b - 1 <= 16 * R) return R;
    return 0;
}

// Position of wavenumber k = k1 + R q in a stored line: complex64 lines keep the q = 2 j and
// 2 j + 1 of a k1 side by side, one 16-byte access of the row pass.
template <bool PAIR>
__host__ __device__ constexpr int rd_pos(int R, int k1, int q) {
    return PAIR ? (q >> 1) * 2 * R + 2 * k1 + (q & 1) : k1 + R * q;
}
// wavenumber stored at position x
template <bool PAIR>
__host__ __device__ constexpr int rd_wavenumber(int R, int x) {
    return PAIR ? (x % (2 * R) >> 1) + R * (2 * (x / (2 * R)) + (x & 1)) : x;
}

// column pass entries: FieldDesc.off field, .ktab table, .rtab slot of the running sum (-1: none)
enum : int { RD_SUM_ONLY = 1 };  // FieldDesc.pad: add the field to the sum and leave it

// One boundary of the row pass: fields 0 and 1, coefficients c[4]: field 0' = c0 f0 + c1 f1, field 1' = c2 f0 + c3 f1
struct RdPair {
    int64_t off0, off1;
    int rt0, rt1;  // tilt/surface tables on the whole grid (-1: none)
    int coef, flags;
};
enum : int { RP_LOAD0 = 1, RP_LOAD1 = 2, RP_STORE0 = 4, RP_STORE1 = 8, RP_ADD1 = 16, RP_ZERO0 = 32 };

template <typename S>
struct RdColArgs {
    cplx<S>* F;
    const FieldDesc* fd;
    int Rx, by;
    const zd* tab;  // [table][My][Mx], or the quarters [table][My/2+1][Mx/2+1]
    int quarter;
    zd* sum;        // [slot][by][Mx]
    const zd* tw;   // exp(-2 pi i t k1 / My) at [k1][t]
};
template <typename S>
struct RdPairArgs {
    cplx<S>* F;
    const RdPair* pairs;
    const zd* coef;
    int by, bx, x0, y0, nx;
    size_t K;
    const zd* rtab;
    const uint32_t* keep;  // [by][16] aperture bits: bit m of entry t for sample t + 16 m
    const zd* tw;          // [k1][t] of Mx
};
// initial fields: the masked window of a source, transformed along x
template <typename S>
struct RdInitArgs {
    cplx<S>* F;
    const FieldDesc* fd;  // .off field, .ktab source index (-1: zero)
    const zd* amp;        // constant sources, or null
    const zd* src;        // [index][ny][nx] sources
    int by, bx, x0, y0, nx;
    size_t K;
    const uint32_t* keep;
    const zd* tw;
    double ex, ey;
    int add;  // add to the stored fields
};
// a sum back to the window, written into whole-grid fields [slot][ny][nx]
struct RdFinalArgs {
    const zd* sum;
    zd* out;
    int by, bx, x0, y0, nx;
    size_t K;
    const zd* tw;
    double ex, ey;
};

template <typename S> void rd_cols(const RdShape& sh, const RdColArgs<S>& a, int nf, hipStream_t s);
template <typename S> void rd_pairs(const RdShape& sh, const RdPairArgs<S>& a, int n, hipStream_t s);
template <typename S> void rd_init(const RdShape& sh, const RdInitArgs<S>& a, int nf, hipStream_t s);
// pair: the sum is of complex64 fields
void rd_final(const RdShape& sh, const RdFinalArgs& a, int n, bool pair, hipStream_t s);
// h [ntab][ny][nx] cut to the window's offsets and made even: out [ntab][My][Mx], times 1/(My Mx)
void rd_crop(const RdShape& sh, const zd* h, int nx, int ny, int ntab, zd* out, hipStream_t s);
// the quarters of ntab tables [My][Mx]
void rd_quarter(const RdShape& sh, const zd* full, int ntab, zd* out, hipStream_t s);
// twiddles [k1 < R][t < 16]
void rd_twiddles(int R, zd* out, hipStream_t s);

}  // namespace bf
