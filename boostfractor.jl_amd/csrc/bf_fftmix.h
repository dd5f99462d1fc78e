// bf_fftmix.h -- register DFTs of R = 4, 5, 6, 8, 10, 12, 16 and 20 points with half of
// their inputs zero or half of their outputs not needed: the passes of the reduced
// propagation's lines of M = 16 R points (bf_reduced.hip).
#pragma once
#include "bf_fftreg.h"

namespace bf {

// exp(-2 pi i m/20) and exp(-2 pi i m/12)
__device__ constexpr double W20R[20] = {
    1.0, 0.951056516295153572116, 0.809016994374947424102, 0.587785252292473129169, 0.309016994374947424102, 0.0,
    -0.309016994374947424102, -0.587785252292473129169, -0.809016994374947424102, -0.951056516295153572116, -1.0,
    -0.951056516295153572116, -0.809016994374947424102, -0.587785252292473129169, -0.309016994374947424102, 0.0,
    0.309016994374947424102, 0.587785252292473129169, 0.809016994374947424102, 0.951056516295153572116};
__device__ constexpr double W20I[20] = {
    0.0, -0.309016994374947424102, -0.587785252292473129169, -0.809016994374947424102, -0.951056516295153572116,
    -1.0, -0.951056516295153572116, -0.809016994374947424102, -0.587785252292473129169, -0.309016994374947424102,
    0.0, 0.309016994374947424102, 0.587785252292473129169, 0.809016994374947424102, 0.951056516295153572116, 1.0,
    0.951056516295153572116, 0.809016994374947424102, 0.587785252292473129169, 0.309016994374947424102};
__device__ constexpr double W12R[12] = {
    1.0, 0.866025403784438646764, 0.5, 0.0, -0.5, -0.866025403784438646764, -1.0, -0.866025403784438646764, -0.5,
    0.0, 0.5, 0.866025403784438646764};
__device__ constexpr double W12I[12] = {
    0.0, -0.5, -0.866025403784438646764, -1.0, -0.866025403784438646764, -0.5, 0.0, 0.5, 0.866025403784438646764,
    1.0, 0.866025403784438646764, 0.5};

// inputs (or outputs) that count: a band of at most (M + 1) / 2 of M = 16 R points, 16 apart per thread
__host__ __device__ constexpr int rd_half(int R) { return (R + 1) / 2; }

// a * exp(-+2 pi i m/R)
template <int R, bool INV>
__device__ __forceinline__ zd twmix(zd a, int m) {
    m %= R;
    if (m == 0) return a;
    double wr, wi;
    if constexpr (20 % R == 0) {
        wr = W20R[m * (20 / R)];
        wi = W20I[m * (20 / R)];
    } else {
        static_assert(12 % R == 0, "unsupported radix");
        wr = W12R[m * (12 / R)];
        wi = W12I[m * (12 / R)];
    }
    if (INV) wi = -wi;
    return cmk<double>(a.re * wr - a.im * wi, a.re * wi + a.im * wr);
}
// +-i s added to and taken from y: the conjugate output pair of an odd DFT
template <bool INV>
__device__ __forceinline__ void pm_i(zd y, zd s, zd& p, zd& q) {  // p = y - i s (forward), q = y + i s
    const zd a = cmk<double>(y.re + s.im, y.im - s.re), b = cmk<double>(y.re - s.im, y.im + s.re);
    p = INV ? b : a;
    q = INV ? a : b;
}
template <bool INV>
__device__ __forceinline__ void dft3(zd& x0, zd& x1, zd& x2) {
    constexpr double S3 = 0.86602540378443864676;
    const zd t = cadd(x1, x2), d = csub(x1, x2);
    const zd y = cmk<double>(fma(-0.5, t.re, x0.re), fma(-0.5, t.im, x0.im)), s = cmk<double>(S3 * d.re, S3 * d.im);
    x0 = cadd(x0, t);
    pm_i<INV>(y, s, x1, x2);
}
template <bool INV>
__device__ __forceinline__ void dft5(zd& x0, zd& x1, zd& x2, zd& x3, zd& x4) {
    constexpr double C1 = 0.30901699437494742410, C2 = -0.80901699437494742410;
    constexpr double S1 = 0.95105651629515357212, S2 = 0.58778525229247312917;
    const zd t1 = cadd(x1, x4), t2 = cadd(x2, x3), d1 = csub(x1, x4), d2 = csub(x2, x3);
    const zd y1 = cmk<double>(fma(C2, t2.re, fma(C1, t1.re, x0.re)), fma(C2, t2.im, fma(C1, t1.im, x0.im)));
    const zd y2 = cmk<double>(fma(C1, t2.re, fma(C2, t1.re, x0.re)), fma(C1, t2.im, fma(C2, t1.im, x0.im)));
    const zd s1 = cmk<double>(fma(S2, d2.re, S1 * d1.re), fma(S2, d2.im, S1 * d1.im));
    const zd s2 = cmk<double>(fma(-S1, d2.re, S2 * d1.re), fma(-S1, d2.im, S2 * d1.im));
    x0 = cmk<double>(x0.re + (t1.re + t2.re), x0.im + (t1.im + t2.im));
    pm_i<INV>(y1, s1, x1, x4);
    pm_i<INV>(y2, s2, x2, x3);
}
template <int Q, bool INV>
__device__ __forceinline__ void dft_odd(zd* d) {
    if constexpr (Q == 3)
        dft3<INV>(d[0], d[1], d[2]);
    else
        dft5<INV>(d[0], d[1], d[2], d[3], d[4]);
}

// DFT of R points, a[m] = 0 for m >= rd_half(R) (not read); natural order in and out
template <int R, bool INV>
__device__ __forceinline__ void dft_in(zd (&a)[R]) {
    constexpr int H = rd_half(R);
    if constexpr (R == 4 || R == 8 || R == 16) {
        dft_reg_m<double, R, INV, (1 << H) - 1, (1 << R) - 1>(a);
    } else if constexpr (R == 5) {
        // x3 = x4 = 0
        a[3] = a[4] = cmk<double>(0, 0);
        dft5<INV>(a[0], a[1], a[2], a[3], a[4]);
    } else {
        // m = Q n1 + n2, k = k1 + P k2: only n1 < P / 2 has inputs
        constexpr int Q = R % 5 == 0 ? 5 : 3, P = R / Q;
        zd b[P][Q];
#pragma unroll
        for (int n2 = 0; n2 < Q; n2++) {
            if constexpr (P == 2) {
                b[0][n2] = a[n2];
                b[1][n2] = a[n2];
            } else {
                zd c0 = a[n2], c1 = a[Q + n2], c2 = cmk<double>(0, 0), c3 = c2;
                radix4m<double, INV, 3, 15>(c0, c1, c2, c3);
                b[0][n2] = c0;
                b[1][n2] = c1;
                b[2][n2] = c2;
                b[3][n2] = c3;
            }
        }
#pragma unroll
        for (int k1 = 0; k1 < P; k1++) {
#pragma unroll
            for (int n2 = 1; n2 < Q; n2++) b[k1][n2] = twmix<R, INV>(b[k1][n2], n2 * k1);
            dft_odd<Q, INV>(b[k1]);
#pragma unroll
            for (int k2 = 0; k2 < Q; k2++) a[k1 + P * k2] = b[k1][k2];
        }
    }
}
// DFT of R points of which the outputs m < rd_half(R) are formed
template <int R, bool INV>
__device__ __forceinline__ void dft_out_half(zd (&a)[R]) {
    constexpr int H = rd_half(R);
    if constexpr (R == 4 || R == 8 || R == 16) {
        dft_reg_m<double, R, INV, (1 << R) - 1, (1 << H) - 1>(a);
    } else if constexpr (R == 5) {
        dft5<INV>(a[0], a[1], a[2], a[3], a[4]);
    } else {
        // inputs k = P n1 + n2, outputs m = m1 + Q m2: only m2 < P / 2 is needed
        constexpr int Q = R % 5 == 0 ? 5 : 3, P = R / Q;
        zd b[P][Q];
#pragma unroll
        for (int n2 = 0; n2 < P; n2++) {
#pragma unroll
            for (int n1 = 0; n1 < Q; n1++) b[n2][n1] = a[P * n1 + n2];
            dft_odd<Q, INV>(b[n2]);
        }
#pragma unroll
        for (int m1 = 0; m1 < Q; m1++) {
#pragma unroll
            for (int n2 = 1; n2 < P; n2++) b[n2][m1] = twmix<R, INV>(b[n2][m1], n2 * m1);
            if constexpr (P == 2) {
                a[m1] = cadd(b[0][m1], b[1][m1]);
            } else {
                radix4m<double, INV, 15, 3>(b[0][m1], b[1][m1], b[2][m1], b[3][m1]);
                a[m1] = b[0][m1];
                a[m1 + Q] = b[1][m1];
            }
        }
    }
}

}  // namespace bf
