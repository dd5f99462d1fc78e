// bf_dft.hip -- the propagation passes with their line transforms on the FP64
// matrix cores (bf_dftmm.h), for lines that are no power of two >= 16.
#include "bf_passes.h"

#include <algorithm>

namespace bf {

// ---------------------------------------------------------------------------
// matrix-core versions of the passes (bf_dftmm.h): FP64 arithmetic, any line
// length up to 1023 that the register transforms do not take.  A block of one
// wave per 16 output indices holds 8 lines.  What bounds them: at 101^2 a bounce
// of 16 frequencies moves 44 MB (the band rows of 224 fields, in and out) and
// issues 2.9e5 MFMAs, 3 us of HBM and 7 us of matrix-core time; the direct sum in
// LDS they replace spent 650 us per bounce on it (LDS reads and 8 n^2 FMAs a line).
// ---------------------------------------------------------------------------
template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_cols_dft(ColArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ unsigned char smem_raw[];
    const int n = a.ny, nx = a.nx, H = n >> 1, ld = dft_ld(n);
    double* E = reinterpret_cast<double*>(smem_raw);
    double* O = E + dft_rows(n, 0) * DFT_LDP;
    double* part = O + dft_rows(n, 0) * DFT_LDP;
    const FieldDesc d = a.fd[blockIdx.y];
    if (a.active && !a.active[d.group]) return;  // uniform over the block
    const int x0 = blockIdx.x * DFT_LINES;
    const int hx = nx / 2, hy = n / 2;
    const uint32_t fl = a.flags;
    const cplx<S>* src = a.src + d.off;
    cplx<S>* dst = a.dst + d.off;
    const zd* kt = d.ktab >= 0 ? a.ktab + (size_t)d.ktab * n * nx : nullptr;
    const bool whole = store_whole(d) || a.all_whole || (fl & (CF_INSHIFT | CF_OUTSHIFT));
    const int band = (fl & (CF_INSHIFT | CF_OUTSHIFT)) ? 0 : dft_fold_lo(n, a.ylo, a.yhi);
    const bool fwd = (fl & CF_FWD) != 0, two = fwd && (fl & CF_INV);
    // fold the input lines (rows outside the band are zero)
    const int base = band & ~3, rows = dft_rows(n, base);
    auto load = [&](int y, int mx) -> zd {
        int sx = mx, sy = y;
        if (fl & CF_INSHIFT) {  // ifftshift on load
            sx = (mx + hx) % nx;
            sy = (y + hy) % n;
        }
        if (!in_band(a, sy)) return cmk<double>(0, 0);
        const size_t o = (size_t)sy * nx + sx;
        zd v = ccast<double>(src[o]);
        if ((fl & CF_KLOAD) && kt) v = cmul(v, ccast<double>(kt[o]));
        return v;
    };
    for (int q = threadIdx.x; q < rows * DFT_LINES; q += blockDim.x) {
        const int c = q & (DFT_LINES - 1), r = q / DFT_LINES, j = base + r, mx = x0 + c;
        const bool ok = mx < nx && j <= H, pr = ok && dft_paired(n, j);
        const zd x = ok ? load(j, mx) : cmk<double>(0, 0);
        const zd m = pr ? load(n - j, mx) : cmk<double>(0, 0);
        if (fwd)
            dft_fold<false>(E, O, r, c, pr, x, m);
        else
            dft_fold<true>(E, O, r, c, pr, x, m);
    }
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    dbl4 e[TPW], o[TPW];
    int tile0, mt = dft_tiles(n, 0), b0 = 0;
    bool own;
    if (two) {
        own = dft_stage<TPW>(E, O, part, n, base, 0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
        // k-space phase of bin k and of its mirror, folded for the inverse
        if (own)
#pragma unroll
            for (int q = 0; q < TPW; q++) {
                const int k = 16 * (tile0 + q * W) + (lane & 15);
                if (tile0 + q * W < mt && k < dft_rows(n, 0)) {
                    const bool pr = dft_paired(n, k);
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const int c = 4 * h + (lane >> 4), mx = x0 + c;
                        const bool ok = mx < nx && k <= H;
                        zd v = ok ? dft_out(e[q], o[q], h) : cmk<double>(0, 0);
                        zd m = pr ? dft_mirror(e[q], o[q], h) : cmk<double>(0, 0);
                        if ((fl & CF_KMID) && kt && ok) {
                            v = cmul(v, ccast<double>(kt[(size_t)k * nx + mx]));
                            if (pr) m = cmul(m, ccast<double>(kt[(size_t)(n - k) * nx + mx]));
                        }
                        dft_fold<true>(E, O, k, c, pr, v, m);
                    }
                }
            }
        b0 = whole ? 0 : band;
        mt = dft_tiles(n, b0);
        own = dft_stage<TPW>(E, O, part, n, 0, b0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    } else {
        b0 = whole || fwd ? 0 : band;
        mt = dft_tiles(n, b0);
        own = dft_stage<TPW>(E, O, part, n, base, b0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    }
    if (!own) return;
    auto store = [&](int y, int mx, zd v) {
        int dx = mx, dy = y;
        if (fl & CF_OUTSHIFT) {  // fftshift on store
            dx = (mx + hx) % nx;
            dy = (y + hy) % n;
        }
        if (whole || in_band(a, dy)) dst[(size_t)dy * nx + dx] = ccast<S>(v);
    };
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = b0 + 16 * (tile0 + q * W) + (lane & 15);
        if (tile0 + q * W >= mt || j > H) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int mx = x0 + 4 * h + (lane >> 4);
            if (mx >= nx) continue;
            store(j, mx, dft_out(e[q], o[q], h));
            if (dft_paired(n, j)) store(n - j, mx, dft_mirror(e[q], o[q], h));
        }
    }
}

template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_rows_dft(RowArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ unsigned char smem_raw[];
    const int n = a.nx, H = n >> 1, ld = dft_ld(n);
    double* E = reinterpret_cast<double*>(smem_raw);
    double* O = E + dft_rows(n, 0) * DFT_LDP;
    double* part = O + dft_rows(n, 0) * DFT_LDP;
    // the grid covers the rows [ylo, yhi) of every field (all rows when yhi <= ylo)
    const bool yband = a.yhi > a.ylo;
    const int nr = yband ? a.yhi - a.ylo : a.ny, y0 = yband ? a.ylo : 0;
    const long nlines = (long)a.nf * nr, line0 = (long)blockIdx.x * DFT_LINES;
    const uint32_t fl = a.flags;
    const bool inv = (fl & RF_INV) != 0, two = inv && (fl & RF_FWD), mask = (fl & RF_MASK) != 0;
    const size_t K = (size_t)n * a.ny;
    // the row's tilt/surface factor and the aperture, after the inverse transform (on load when there is none)
    auto middle = [&](const FieldDesc& d, int y, int x, zd v) -> zd {
        if ((fl & RF_RTAB) && d.rtab >= 0) v = cmul(v, ccast<double>(a.rtab[(size_t)d.rtab * K + (size_t)y * n + x]));
        if (mask && !in_aperture(a.X[x], a.Y[y], a.R2)) v = cmk<double>(0, 0);
        return v;
    };
    const int a0 = !inv && mask ? a.dft.lo & ~3 : 0, rows = dft_rows(n, a0);
    for (int q = threadIdx.x; q < rows * DFT_LINES; q += blockDim.x) {
        const int c = q / rows, r = q - c * rows, j = a0 + r;
        const long l = line0 + c;
        bool ok = l < nlines && j <= H;
        zd x = cmk<double>(0, 0), m = x;
        const bool pr = dft_paired(n, j);
        if (ok) {
            const FieldDesc d = a.fd[l / nr];
            const int y = y0 + (int)(l % nr);
            if (!a.active || a.active[d.group]) {
                const cplx<S>* row = a.base + d.off + (size_t)y * n;
                x = ccast<double>(row[j]);
                if (pr) m = ccast<double>(row[n - j]);
                if (!inv) {
                    x = middle(d, y, j, x);
                    if (pr) m = middle(d, y, n - j, m);
                }
            }
        }
        if (inv)
            dft_fold<true>(E, O, r, c, pr && ok, x, m);
        else
            dft_fold<false>(E, O, r, c, pr && ok, x, m);
    }
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    // this lane's two lines
    FieldDesc d[2];
    int y[2];
    bool ok[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const long l = line0 + 4 * h + (lane >> 4);
        ok[h] = l < nlines;
        d[h] = a.fd[ok[h] ? l / nr : 0];
        y[h] = y0 + (int)(ok[h] ? l % nr : 0);
        if (a.active && !a.active[d[h].group]) ok[h] = false;
    }
    dbl4 e[TPW], o[TPW];
    int tile0, b0 = two && mask ? a.dft.lo : 0, mt = dft_tiles(n, b0);
    bool own = dft_stage<TPW>(E, O, part, n, a0, b0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    if (two) {
        const int a2 = b0 & ~3;  // the mask zeroes the folded indices below b0
        if (own)
#pragma unroll
            for (int q = 0; q < TPW; q++) {
                const int j = b0 + 16 * (tile0 + q * W) + (lane & 15);
                if (tile0 + q * W >= mt || j > H) continue;
                const bool pr = dft_paired(n, j);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const zd v = middle(d[h], y[h], j, dft_out(e[q], o[q], h));
                    const zd m = pr ? middle(d[h], y[h], n - j, dft_mirror(e[q], o[q], h)) : cmk<double>(0, 0);
                    dft_fold<false>(E, O, j - a2, 4 * h + (lane >> 4), pr, v, m);
                }
            }
        dft_zero_rows(E, O, 0, b0 - a2);
        dft_zero_rows(E, O, H + 1 - a2, dft_rows(n, a2));
        b0 = 0;
        mt = dft_tiles(n, 0);
        own = dft_stage<TPW>(E, O, part, n, a2, 0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    }
    if (!own) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = b0 + 16 * (tile0 + q * W) + (lane & 15);
        if (tile0 + q * W >= mt || j > H) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (!ok[h]) continue;
            cplx<S>* row = a.base + d[h].off + (size_t)y[h] * n;
            zd v = dft_out(e[q], o[q], h), m = dft_mirror(e[q], o[q], h);
            const bool pr = dft_paired(n, j), mid = inv && !two;
            row[j] = ccast<S>(mid ? middle(d[h], y[h], j, v) : v);
            if (pr) row[n - j] = ccast<S>(mid ? middle(d[h], y[h], n - j, m) : m);
        }
    }
}

// The fused row pass of a bounce: 4 rows of the two fields that meet at boundary
// b, lines 0..3 the right-moving ones (A) and 4..7 the left-moving ones (B), so
// that a lane holds A and B of one row at an output index and at its mirror.
template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_dancer_rows_dft(DancerRowArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ unsigned char smem_raw[];
    __shared__ double red[16];
    const int n = a.nx, H = n >> 1, ld = dft_ld(n);
    double* E = reinterpret_cast<double*>(smem_raw);
    double* O = E + dft_rows(n, 0) * DFT_LDP;
    double* part = O + dft_rows(n, 0) * DFT_LDP;
    const int f = blockIdx.y;
    int b, tile;
    bool exit_only;
    dancer_block(a, blockIdx.x, b, tile, exit_only);
    if (a.active && !a.active[f]) return;  // uniform over the block
    if (a.count && blockIdx.x == 0 && threadIdx.x == 0) a.count[f] += 1;
    const size_t K = (size_t)n * a.ny;
    const int y0 = tile * 4;
    const bool hasA = b > 0, hasB = b < a.R;
    cplx<S>* FA = a.fields + (((size_t)f * a.R + (hasA ? b - 1 : 0)) * 2 + a.rm) * K;
    cplx<S>* FB = a.fields + (((size_t)f * a.R + (hasB ? b : 0)) * 2 + (1 - a.rm)) * K;
    const int rows = dft_rows(n, 0);
    for (int q = threadIdx.x; q < rows * DFT_LINES; q += blockDim.x) {
        const int c = q / rows, j = q - c * rows, y = y0 + (c & 3);
        const bool ok = (c < 4 ? hasA : hasB) && y < a.ny && j <= H, pr = dft_paired(n, j);
        const cplx<S>* row = (c < 4 ? FA : FB) + (size_t)y * n;
        const zd x = ok ? ccast<double>(row[j]) : cmk<double>(0, 0);
        const zd m = ok && pr ? ccast<double>(row[n - j]) : cmk<double>(0, 0);
        dft_fold<true>(E, O, j, c, pr, x, m);
    }
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int y = y0 + (lane >> 4);
    const bool oky = y < a.ny;
    const double yy = a.Y[oky ? y : 0];
    const bool fwd = (a.flags & DF_FWD) != 0;
    const int lo = fwd ? a.dft.lo : 0;  // the next aperture keeps the folded indices >= lo
    const int b0 = (b == a.R || (a.flags & DF_AMAX)) ? 0 : lo, a2 = lo & ~3;
    int tile0, mt = dft_tiles(n, b0);
    dbl4 e[TPW], o[TPW];
    bool own = dft_stage<TPW>(E, O, part, n, 0, b0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    // boundary update (src/boost_fractor_recurprop.jl:90-119)
    const zd r = a.coef[b];
    const zd omr = cmk<double>(1.0 - r.re, -r.im), opr = cmk<double>(1.0 + r.re, r.im), mr = cmk<double>(-r.re, -r.im);
    const int tA = a.rtab && hasA ? a.rtab_idx[f * a.R + b - 1] : -1, tB = a.rtab && hasB ? a.rtab_idx[f * a.R + b] : -1;
    double vmax = 0.0;
    auto update = [&](int x, zd& A, zd& B) {
        const size_t p = (size_t)y * n + x;
        if (tA >= 0) A = cmul(A, ccast<double>(a.rtab[(size_t)tA * K + p]));
        if (tB >= 0) B = cmul(B, ccast<double>(a.rtab[(size_t)tB * K + p]));
        zd nA, nB;
        if (b == a.R) {  // exit boundary: Eout += (1+r) A, A' = r A
            zd* eo = a.Eout + (size_t)f * a.eout_fstride + (size_t)a.slice * K + p;
            const zd v = cmul(opr, A);
            *eo = (a.flags & DF_EOUT_ASSIGN) ? v : cadd(*eo, v);
            nA = cmul(A, r);
        } else {  // A' = r A + (1-r) B
            nA = cadd(cmul(A, r), cmul(omr, B));
        }
        // mirror: B' = -r B; else B' = -r B + (1+r) A
        nB = b == 0 ? cmul(B, mr) : cadd(cmul(B, mr), cmul(opr, A));
        A = hasA ? nA : cmk<double>(0, 0);
        B = hasB ? nB : cmk<double>(0, 0);
        if (a.flags & DF_AMAX) vmax = fmax(vmax, fmax(hypot(A.re, A.im), hypot(B.re, B.im)));
        if (fwd && !in_aperture(a.X[x], yy, a.R2)) A = B = cmk<double>(0, 0);  // next bounce's aperture
    };
    if (own && oky)
#pragma unroll
        for (int q = 0; q < TPW; q++) {
            const int j = b0 + 16 * (tile0 + q * W) + (lane & 15);
            if (tile0 + q * W >= mt || j > H) continue;
            const bool pr = dft_paired(n, j);
            zd A = dft_out(e[q], o[q], 0), B = dft_out(e[q], o[q], 1);
            zd mA = dft_mirror(e[q], o[q], 0), mB = dft_mirror(e[q], o[q], 1);
            update(j, A, B);
            if (pr) update(n - j, mA, mB);
            if (j >= lo) {
                dft_fold<false>(E, O, j - a2, lane >> 4, pr, A, mA);
                dft_fold<false>(E, O, j - a2, 4 + (lane >> 4), pr, B, mB);
            }
        }
    if (a.flags & DF_AMAX) {
        for (int w = 32; w > 0; w >>= 1) vmax = fmax(vmax, __shfl_xor(vmax, w));
        if (lane == 0) red[threadIdx.x >> 6] = vmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            double m = 0.0;
            for (int w = 0; w < W; w++) m = fmax(m, red[w]);
            if (m > 0.0) atomic_max_pos(a.amax + f, m);
        }
    }
    if (!fwd || exit_only) return;  // only Eout is needed
    dft_zero_rows(E, O, 0, lo - a2);
    dft_zero_rows(E, O, H + 1 - a2, dft_rows(n, a2));
    mt = dft_tiles(n, 0);
    own = dft_stage<TPW>(E, O, part, n, a2, 0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    if (!own || !oky) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = 16 * (tile0 + q * W) + (lane & 15);
        if (tile0 + q * W >= mt || j > H) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (!(h == 0 ? hasA : hasB)) continue;
            cplx<S>* row = (h == 0 ? FA : FB) + (size_t)y * n;
            row[j] = ccast<S>(dft_out(e[q], o[q], h));
            if (dft_paired(n, j)) row[n - j] = ccast<S>(dft_mirror(e[q], o[q], h));
        }
    }
}

// The pair step on the matrix cores: 4 rows, lines 0..3 field i, 4..7 field i+1
template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_ch_pair_dft(ChPairArgs<T> a, int n) {
    using S = typename Storage<T>::type;
    extern __shared__ unsigned char smem_raw[];
    const int H = n >> 1, ld = dft_ld(n);
    double* E = reinterpret_cast<double*>(smem_raw);
    double* O = E + dft_rows(n, 0) * DFT_LDP;
    double* part = O + dft_rows(n, 0) * DFT_LDP;
    const int en = blockIdx.y;
    const FieldDesc d0 = a.fd[2 * en], d1 = a.fd[2 * en + 1];
    if (a.active && !a.active[d0.group]) return;  // uniform over the block
    const size_t K = (size_t)n * a.ny;
    const int y0 = a.ylo + blockIdx.x * 4;
    cplx<S>* F0 = a.F + d0.off;
    cplx<S>* F1 = a.F + d1.off;
    const int rows = dft_rows(n, 0);
    for (int q = threadIdx.x; q < rows * DFT_LINES; q += blockDim.x) {
        const int c = q / rows, j = q - c * rows, y = y0 + (c & 3);
        const bool ok = y < a.yhi && j <= H, pr = dft_paired(n, j);
        const cplx<S>* row = (c < 4 ? F0 : F1) + (size_t)y * n;
        const zd x = ok ? ccast<double>(row[j]) : cmk<double>(0, 0);
        const zd m = ok && pr ? ccast<double>(row[n - j]) : cmk<double>(0, 0);
        dft_fold<true>(E, O, j, c, pr, x, m);
    }
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int y = y0 + (lane >> 4);
    const bool oky = y < a.yhi;
    const double yy = a.Y[oky ? y : 0];
    const bool xout = a.xout != 0;
    const int lo = xout ? a.dft.lo : 0, a2 = lo & ~3;  // the mask of the next transform keeps the folded indices >= lo
    int tile0, mt = dft_tiles(n, lo);
    dbl4 e[TPW], o[TPW];
    bool own = dft_stage<TPW>(E, O, part, n, 0, lo, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    const zd* cf = a.coef + 4 * (d0.pad >> FD_PAIR_SHIFT);
    const zd rl = cf[0], tr = cf[1], rr = cf[2], tl = cf[3];
    const int t0 = a.rtab ? d0.rtab : -1, t1 = a.rtab ? d1.rtab : -1;
    // k_ch_pair: Fn = c rl + tr a, Fi = a rr + tl c (a: field i, c: field i+1), rounded as they are stored
    auto update = [&](int x, zd& A, zd& B) {
        const size_t p = (size_t)y * n + x;
        if (t0 >= 0) A = cmul(A, ccast<double>(a.rtab[(size_t)t0 * K + p]));
        if (t1 >= 0) B = cmul(B, ccast<double>(a.rtab[(size_t)t1 * K + p]));
        A = ccast<double>(ccast<S>(A));
        B = ccast<double>(ccast<S>(B));
        const zd nA = cadd(cmul(A, rr), cmul(tl, B)), nB = cadd(cmul(B, rl), cmul(tr, A));
        A = ccast<double>(ccast<S>(nA));
        B = ccast<double>(ccast<S>(nB));
        if (xout && !in_aperture(a.X[x], yy, a.R2)) A = B = cmk<double>(0, 0);
    };
    if (own && oky)
#pragma unroll
        for (int q = 0; q < TPW; q++) {
            const int j = lo + 16 * (tile0 + q * W) + (lane & 15);
            if (tile0 + q * W >= mt || j > H) continue;
            const bool pr = dft_paired(n, j);
            zd A = dft_out(e[q], o[q], 0), B = dft_out(e[q], o[q], 1);
            zd mA = dft_mirror(e[q], o[q], 0), mB = dft_mirror(e[q], o[q], 1);
            update(j, A, B);
            if (pr) update(n - j, mA, mB);
            if (xout) {
                dft_fold<false>(E, O, j - a2, lane >> 4, pr, A, mA);
                dft_fold<false>(E, O, j - a2, 4 + (lane >> 4), pr, B, mB);
            } else {
                cplx<S>* r0 = F0 + (size_t)y * n;
                cplx<S>* r1 = F1 + (size_t)y * n;
                r0[j] = ccast<S>(A);
                r1[j] = ccast<S>(B);
                if (pr) {
                    r0[n - j] = ccast<S>(mA);
                    r1[n - j] = ccast<S>(mB);
                }
            }
        }
    if (!xout) return;
    dft_zero_rows(E, O, 0, lo - a2);
    dft_zero_rows(E, O, H + 1 - a2, dft_rows(n, a2));
    mt = dft_tiles(n, 0);
    own = dft_stage<TPW>(E, O, part, n, a2, 0, mt, a.dft.smax, a.dft.tab, ld, e, o, tile0);
    if (!own || !oky) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = 16 * (tile0 + q * W) + (lane & 15);
        if (tile0 + q * W >= mt || j > H) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            cplx<S>* row = (h == 0 ? F0 : F1) + (size_t)y * n;
            row[j] = ccast<S>(dft_out(e[q], o[q], h));
            if (dft_paired(n, j)) row[n - j] = ccast<S>(dft_mirror(e[q], o[q], h));
        }
    }
}

// Launch shape of the matrix-core passes for lines of n points: a wave per 16
// output indices (two tiles per wave beyond 16 waves), the planes of all folded
// rows, and room for the partial tiles of a shared contraction while the block
// stays within the 160 KB of a CU.
struct DftShape {
    int waves, tpw, smax;
    size_t smem;
    explicit DftShape(int n) {
        const int mt = dft_tiles(n, 0);
        tpw = mt <= 16 ? 1 : 2;
        waves = (mt + tpw - 1) / tpw;
        if (waves > 2) waves = (waves + 3) & ~3;  // whole rounds over the four SIMDs
        const size_t planes = sizeof(double) * 2 * DFT_LDP * (size_t)dft_rows(n, 0);
        const size_t part = sizeof(double) * DFT_PART * (size_t)(waves - 1);
        const bool share = planes + part <= 152 * 1024;
        smax = share ? 4 : 1;
        smem = planes + (share ? part : 0);
    }
};
#define BF_DFT_LAUNCH(kernel, T, sh, grid, s, ...)                                                                  \
    do {                                                                                                             \
        if ((sh).tpw == 1) {                                                                                         \
            allow_lds((const void*)kernel<T, 1>, (sh).smem);                                                         \
            hipLaunchKernelGGL((kernel<T, 1>), grid, dim3(64 * (sh).waves), (sh).smem, s, __VA_ARGS__);              \
        } else {                                                                                                     \
            allow_lds((const void*)kernel<T, 2>, (sh).smem);                                                         \
            hipLaunchKernelGGL((kernel<T, 2>), grid, dim3(64 * (sh).waves), (sh).smem, s, __VA_ARGS__);              \
        }                                                                                                            \
        BF_CHECK_LAUNCH();                                                                                           \
    } while (0)

template <typename T>
void launch_rows_dft(RowArgs<T> a, hipStream_t s) {
    const DftShape sh(a.nx);
    a.dft.smax = sh.smax;
    const long nlines = (long)a.nf * (a.yhi > a.ylo ? a.yhi - a.ylo : a.ny);
    BF_DFT_LAUNCH(k_rows_dft, T, sh, dim3((unsigned)((nlines + DFT_LINES - 1) / DFT_LINES)), s, a);
}
template <typename T>
void launch_cols_dft(ColArgs<T> a, hipStream_t s) {
    const DftShape sh(a.ny);
    a.dft.smax = sh.smax;
    BF_DFT_LAUNCH(k_cols_dft, T, sh, dim3((a.nx + DFT_LINES - 1) / DFT_LINES, a.nf), s, a);
}
template <typename T>
void launch_dancer_rows_dft(DancerRowArgs<T> a, int fb, hipStream_t s) {
    const DftShape sh(a.nx);
    a.dft.smax = sh.smax;
    const unsigned nblk = dancer_tiles(a, 4);
    BF_DFT_LAUNCH(k_dancer_rows_dft, T, sh, dim3(nblk, fb), s, a);
}
template <typename T>
void launch_ch_pair_dft(ChPairArgs<T> a, int nx, int entries, hipStream_t s) {
    if (!a.dft.tab) throw std::runtime_error("the pair step's row transforms have no table");
    const DftShape sh(nx);
    a.dft.smax = sh.smax;
    BF_DFT_LAUNCH(k_ch_pair_dft, T, sh, dim3((a.yhi - a.ylo + 3) / 4, entries), s, a, nx);
}
#define BF_DFT_INSTANCES(T)                                                     \
    template void launch_rows_dft<T>(RowArgs<T>, hipStream_t);                  \
    template void launch_cols_dft<T>(ColArgs<T>, hipStream_t);                  \
    template void launch_dancer_rows_dft<T>(DancerRowArgs<T>, int, hipStream_t); \
    template void launch_ch_pair_dft<T>(ChPairArgs<T>, int, int, hipStream_t);
BF_DFT_INSTANCES(double)
BF_DFT_INSTANCES(float)

// (cos, sin)(2 pi a b / n) for the matrix-core line transforms, a, b < dft_ld(n)
__global__ void k_dft_table(double2* out, int n, int ld) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ld * ld; i += gridDim.x * blockDim.x) {
        const int m = (int)(((long)(i / ld) * (i % ld)) % n);
        double s, c;
        sincospi(2.0 * (double)m / (double)n, &s, &c);
        out[i] = make_double2(c, s);
    }
}
// The context keeps the tables of the last lengths used (at most 4.4 MB each, n = 1023); an
// engine holds its own reference, so a table dropped here lives as long as a plan that reads it.
std::shared_ptr<DevBuf> dft_table(bf_ctx* ctx, int n) {
    auto& cache = ctx->dft_tables;
    for (size_t q = 0; q < cache.size(); q++)
        if (cache[q].first == n) {
            std::rotate(cache.begin() + q, cache.begin() + q + 1, cache.end());
            return cache.back().second;
        }
    const int ld = dft_ld(n);
    auto b = std::make_shared<DevBuf>(sizeof(double2) * (size_t)ld * ld);
    hipLaunchKernelGGL(k_dft_table, dim3((ld * ld + 255) / 256), dim3(256), 0, ctx->stream, b->as<double2>(), n, ld);
    BF_CHECK_LAUNCH();
    if (cache.size() >= 8) cache.erase(cache.begin());
    cache.emplace_back(n, b);
    return b;
}

}  // namespace bf
