// bf_dft.hip -- the propagation passes with their line transforms on the FP64
// matrix cores (bf_dftmm.h), for lines that are no power of two >= 16.
#include "bf_passes.h"

#include <algorithm>

namespace bf {

// ---------------------------------------------------------------------------
// matrix-core versions of the passes (bf_dftmm.h): FP64 arithmetic, any line
// length up to 1023 that the register transforms do not take.  A block of one
// wave per 16 output indices holds 8 lines.  What bounds them: a bounce of 16
// frequencies and 3 disks at 101^2 moves 44 MB (the band rows of 224 fields, in
// and out) and issues 3.2e5 MFMAs, 8 us of HBM and 9 us of matrix-core time; the
// column pass takes 27 us and the row pass 19 us, in chains of dependent loads
// (kernel arguments, descriptor, lines, output) with 4 waves per SIMD.  The
// direct sums in LDS that they replace took 458 and 193 us (8 n^2 FMAs a line and
// an LDS read for each).  Loads predicated by an out-of-range buffer offset
// instead of branches, the sine and the cosine product of a shared tile in waves
// of their own, and the tables' loads issued before the first wait brought them
// from 38 and 25 us.
// ---------------------------------------------------------------------------
// FL != 0: the flags are fixed at compile time (the solvers' FWD|KMID|INV, no shifts)
template <typename T, int TPW, uint32_t FL>
__global__ void __launch_bounds__(1024) k_cols_dft(ColArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ double2 dft_smem[];
    const int n = a.ny, nx = a.nx, H = n >> 1;
    double2* P = dft_smem;
    double2* part = P + dft_rows(n, 0) * DFT_LDP;
    const FieldDesc d = a.fd[blockIdx.y];
    const bool idle = a.active && !a.active[d.group];  // uniform over the block
    const int W = blockDim.x >> 6, lane = threadIdx.x & 63;
    const int x0 = blockIdx.x * DFT_LINES;
    constexpr uint32_t PROP = CF_FWD | CF_KMID | CF_INV, SZ = sizeof(cplx<S>);
    const uint32_t fl = FL ? FL : a.flags;
    dbl4 e[TPW], o[TPW];
    if constexpr (FL == PROP) {
        // A resource over the band rows answers the others with zero, as one over the
        // k-space table answers bins without a mirror: no branch on either
        const bool whole = store_whole(d) || a.all_whole;
        const int band = dft_fold_lo(n, a.ylo, a.yhi), base = band & ~3, rows = dft_rows(n, base);
        const uint32_t rowb = (uint32_t)nx * SZ, bandb = (uint32_t)(a.yhi - a.ylo) * rowb;
        const auto rs = buf_rsrc(a.src + d.off + (size_t)a.ylo * nx, bandb);
        const uint32_t KT = (uint32_t)n * (uint32_t)nx * (uint32_t)sizeof(zd), krow = (uint32_t)nx * (uint32_t)sizeof(zd);
        const auto rk = buf_rsrc(a.ktab + (size_t)d.ktab * n * nx, KT);
        int mt = dft_tiles(n, 0);
        const DftShare s1(mt, a.dft.smax);
        // The field's and the phase table's loads go out together, before anything waits:
        // a dependent load costs ~1 us here, more than the products of a stage.
        const int c = threadIdx.x & 7, r0 = threadIdx.x >> 3, rstep = blockDim.x >> 3;
        const uint32_t cb = (uint32_t)(x0 + c) * SZ - (uint32_t)a.ylo * rowb;
        auto point = [&](int r, cplx<S>& x, cplx<S>& m) {
            const int j = base + r;
            const bool in = x0 + c < nx && j <= H;
            x = buf_load<S>(rs, in ? cb + (uint32_t)j * rowb : BUF_OOB);
            m = buf_load<S>(rs, in && j > 0 && 2 * j < n ? cb + (uint32_t)(n - j) * rowb : BUF_OOB);
        };
        cplx<S> x, m;
        point(r0, x, m);
        zd pv[TPW][2], pm[TPW][2];
#pragma unroll
        for (int q = 0; q < TPW; q++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int mx = x0 + 4 * h + (lane >> 4), k = 16 * (s1.first + q * W) + (lane & 15);
                const bool in = mx < nx && k <= H && s1.s == 0;
                const uint32_t kb = (uint32_t)mx * (uint32_t)sizeof(zd);
                pv[q][h] = buf_load<double>(rk, in ? kb + (uint32_t)k * krow : BUF_OOB);
                pm[q][h] = buf_load<double>(rk, in && k > 0 && 2 * k < n ? kb + (uint32_t)(n - k) * krow : BUF_OOB);
            }
        if (idle) return;
        for (int r = r0; r < rows; r += rstep) {
            if (r != r0) point(r, x, m);
            dft_fold<false>(P, r, c, ccast<double>(x), ccast<double>(m));
        }
        dft_stage<TPW>(P, part, n, base, 0, mt, s1, a.dft.tab, e, o);
        // k-space phase of bin k and of its mirror, folded for the inverse
        if (s1.own(mt))
#pragma unroll
            for (int q = 0; q < TPW; q++) {
                const int k = 16 * (s1.first + q * W) + (lane & 15);
                if (s1.first + q * W < mt && k < dft_rows(n, 0))
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        dft_fold<true>(P, k, 4 * h + (lane >> 4), cmul(dft_out(e[q], o[q], h), pv[q][h]),
                                       cmul(dft_mirror(e[q], o[q], h), pm[q][h]));
            }
        const int b0 = whole ? 0 : band;
        mt = dft_tiles(n, b0);
        const DftShare s2(mt, a.dft.smax);
        dft_stage<TPW>(P, part, n, 0, b0, mt, s2, a.dft.tab, e, o);
        if (!s2.own(mt)) return;
        // band rows, or every row of a field stored whole
        const int s0 = whole ? 0 : a.ylo;
        const auto rd = buf_rsrc(a.dst + d.off + (size_t)s0 * nx, whole ? (uint32_t)n * rowb : bandb);
#pragma unroll
        for (int q = 0; q < TPW; q++) {
            const int j = b0 + 16 * (s2.first + q * W) + (lane & 15);
            if (s2.first + q * W >= mt) continue;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int mx = x0 + 4 * h + (lane >> 4);
                const bool in = mx < nx && j <= H;
                const uint32_t cb = (uint32_t)mx * SZ - (uint32_t)s0 * rowb;
                buf_store<S>(rd, in ? cb + (uint32_t)j * rowb : BUF_OOB, ccast<S>(dft_out(e[q], o[q], h)));
                buf_store<S>(rd, in && j > 0 && 2 * j < n ? cb + (uint32_t)(n - j) * rowb : BUF_OOB,
                             ccast<S>(dft_mirror(e[q], o[q], h)));
            }
        }
        return;
    }
    if (idle) return;
    // one transform, or shifted loads and stores (momentum space): every row
    const int hx = nx / 2, hy = n / 2;
    const cplx<S>* src = a.src + d.off;
    cplx<S>* dst = a.dst + d.off;
    const zd* kt = d.ktab >= 0 ? a.ktab + (size_t)d.ktab * n * nx : nullptr;
    const bool fwd = (fl & CF_FWD) != 0, two = fwd && (fl & CF_INV);
    auto load = [&](int y, int mx) -> zd {
        int sx = mx, sy = y;
        if (fl & CF_INSHIFT) {  // ifftshift on load
            sx = (mx + hx) % nx;
            sy = (y + hy) % n;
        }
        if (!in_band(a, sy)) return cmk<double>(0, 0);
        const size_t p = (size_t)sy * nx + sx;
        zd v = ccast<double>(src[p]);
        if ((fl & CF_KLOAD) && kt) v = cmul(v, ccast<double>(kt[p]));
        return v;
    };
    for (int q = threadIdx.x; q < dft_rows(n, 0) * DFT_LINES; q += blockDim.x) {
        const int c = q & (DFT_LINES - 1), j = q / DFT_LINES, mx = x0 + c;
        const bool ok = mx < nx && j <= H;
        const zd x = ok ? load(j, mx) : cmk<double>(0, 0);
        const zd m = ok && dft_paired(n, j) ? load(n - j, mx) : cmk<double>(0, 0);
        if (fwd)
            dft_fold<false>(P, j, c, x, m);
        else
            dft_fold<true>(P, j, c, x, m);
    }
    const int mt = dft_tiles(n, 0);
    const DftShare sh(mt, a.dft.smax);
    dft_stage<TPW>(P, part, n, 0, 0, mt, sh, a.dft.tab, e, o);
    if (two) {
        if (sh.own(mt))
#pragma unroll
            for (int q = 0; q < TPW; q++) {
                const int k = 16 * (sh.first + q * W) + (lane & 15);
                if (sh.first + q * W < mt && k < dft_rows(n, 0)) {
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
                        dft_fold<true>(P, k, c, v, m);
                    }
                }
            }
        dft_stage<TPW>(P, part, n, 0, 0, mt, sh, a.dft.tab, e, o);
    }
    if (!sh.own(mt)) return;
    const bool whole = store_whole(d) || a.all_whole;
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
        const int j = 16 * (sh.first + q * W) + (lane & 15);
        if (sh.first + q * W >= mt || j > H) continue;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int mx = x0 + 4 * h + (lane >> 4);
            if (mx >= nx) continue;
            store(j, mx, dft_out(e[q], o[q], h));
            if (dft_paired(n, j)) store(n - j, mx, dft_mirror(e[q], o[q], h));
        }
    }
}

// Loads and folds line `c` of the block (one wave per line, lanes along it) from
// its first element p; null: a zero line.  map(x, v): value of element x.
template <bool INV, typename S, typename F>
__device__ __forceinline__ void dft_load_line(double2* P, int n, int base, int c, const cplx<S>* p, F map) {
    const int lane = threadIdx.x & 63, rows = dft_rows(n, base);
    const auto r = buf_rsrc(p, p ? (uint32_t)n * (uint32_t)sizeof(cplx<S>) : 0u);
    for (int q = lane; q < rows; q += 64) {
        const int j = base + q;
        const bool in = j <= n >> 1, pr = in && j > 0 && 2 * j < n;
        const cplx<S> x = buf_load<S>(r, in ? (uint32_t)j * (uint32_t)sizeof(cplx<S>) : BUF_OOB);
        const cplx<S> m = buf_load<S>(r, pr ? (uint32_t)(n - j) * (uint32_t)sizeof(cplx<S>) : BUF_OOB);
        dft_fold<INV>(P, q, c, map(in ? j : 0, ccast<double>(x)), map(pr ? n - j : 0, ccast<double>(m)));
    }
}

template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_rows_dft(RowArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ double2 dft_smem[];
    const int n = a.nx, H = n >> 1;
    double2* P = dft_smem;
    double2* part = P + dft_rows(n, 0) * DFT_LDP;
    // the grid covers the rows [ylo, yhi) of every field (all rows when yhi <= ylo)
    const bool yband = a.yhi > a.ylo;
    const int nr = yband ? a.yhi - a.ylo : a.ny, y0 = yband ? a.ylo : 0;
    const int nlines = a.nf * nr, line0 = blockIdx.x * DFT_LINES;
    const uint32_t fl = a.flags;
    const bool inv = (fl & RF_INV) != 0, two = inv && (fl & RF_FWD), mask = (fl & RF_MASK) != 0;
    const size_t K = (size_t)n * a.ny;
    // the row's tilt/surface factor and the aperture, after the inverse transform (on load when there is none)
    auto middle = [&](const FieldDesc& d, int y, int x, zd v) -> zd {
        if ((fl & RF_RTAB) && d.rtab >= 0) v = cmul(v, ccast<double>(a.rtab[(size_t)d.rtab * K + (size_t)y * n + x]));
        if (mask && !in_aperture(a.X[x], a.Y[y], a.R2)) v = cmk<double>(0, 0);
        return v;
    };
    const int a0 = !inv && mask ? a.dft.lo & ~3 : 0;
    const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int c = wave; c < DFT_LINES; c += W) {
        const int l = line0 + c;
        const FieldDesc d = a.fd[l < nlines ? l / nr : 0];
        const int y = y0 + (l < nlines ? l % nr : 0);
        const bool ok = l < nlines && (!a.active || a.active[d.group]);
        const cplx<S>* p = ok ? a.base + d.off + (size_t)y * n : nullptr;
        if (inv)
            dft_load_line<true>(P, n, a0, c, p, [](int, zd v) { return v; });
        else
            dft_load_line<false>(P, n, a0, c, p, [&](int x, zd v) { return middle(d, y, x, v); });
    }
    // this lane's two lines
    FieldDesc d[2];
    int y[2];
    bool ok[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int l = line0 + 4 * h + (lane >> 4);
        ok[h] = l < nlines;
        d[h] = a.fd[ok[h] ? l / nr : 0];
        y[h] = y0 + (ok[h] ? l % nr : 0);
        if (a.active && !a.active[d[h].group]) ok[h] = false;
    }
    dbl4 e[TPW], o[TPW];
    int b0 = two && mask ? a.dft.lo : 0, mt = dft_tiles(n, b0);
    DftShare sh(mt, a.dft.smax);
    dft_stage<TPW>(P, part, n, a0, b0, mt, sh, a.dft.tab, e, o);
    if (two) {
        const int a2 = b0 & ~3;  // the mask zeroes the folded indices below b0
        if (sh.own(mt))
#pragma unroll
            for (int q = 0; q < TPW; q++) {
                const int j = b0 + 16 * (sh.first + q * W) + (lane & 15);
                if (sh.first + q * W >= mt || j > H) continue;
                const bool pr = dft_paired(n, j);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const zd v = middle(d[h], y[h], j, dft_out(e[q], o[q], h));
                    const zd m = pr ? middle(d[h], y[h], n - j, dft_mirror(e[q], o[q], h)) : cmk<double>(0, 0);
                    dft_fold<false>(P, j - a2, 4 * h + (lane >> 4), v, m);
                }
            }
        dft_zero_rows(P, 0, b0 - a2);
        dft_zero_rows(P, H + 1 - a2, dft_rows(n, a2));
        b0 = 0;
        mt = dft_tiles(n, 0);
        sh = DftShare(mt, a.dft.smax);
        dft_stage<TPW>(P, part, n, a2, 0, mt, sh, a.dft.tab, e, o);
    }
    if (!sh.own(mt)) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = b0 + 16 * (sh.first + q * W) + (lane & 15);
        if (sh.first + q * W >= mt || j > H) continue;
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
    extern __shared__ double2 dft_smem[];
    __shared__ double red[16];
    const int n = a.nx, H = n >> 1;
    double2* P = dft_smem;
    double2* part = P + dft_rows(n, 0) * DFT_LDP;
    const int f = blockIdx.y;
    int b, tile;
    bool exit_only;
    dancer_block(a, blockIdx.x, b, tile, exit_only);
    const bool idle = a.active && !a.active[f];  // uniform over the block
    const size_t K = (size_t)n * a.ny;
    const int y0 = tile * 4;
    const bool hasA = b > 0, hasB = b < a.R;
    cplx<S>* FA = a.fields + (((size_t)f * a.R + (hasA ? b - 1 : 0)) * 2 + a.rm) * K;
    cplx<S>* FB = a.fields + (((size_t)f * a.R + (hasB ? b : 0)) * 2 + (1 - a.rm)) * K;
    const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int c = wave; c < DFT_LINES; c += W) {
        const int yl = y0 + (c & 3);
        const bool ok = (c < 4 ? hasA : hasB) && yl < a.ny;
        dft_load_line<true>(P, n, 0, c, ok ? (c < 4 ? FA : FB) + (size_t)yl * n : nullptr, [](int, zd v) { return v; });
    }
    if (idle) return;  // (the lines were loaded meanwhile)
    if (a.count && blockIdx.x == 0 && threadIdx.x == 0) a.count[f] += 1;
    const int y = y0 + (lane >> 4);
    const bool oky = y < a.ny;
    const double yy = a.Y[oky ? y : 0];
    const bool fwd = (a.flags & DF_FWD) != 0;
    const int lo = fwd ? a.dft.lo : 0;  // the next aperture keeps the folded indices >= lo
    const int b0 = (b == a.R || (a.flags & DF_AMAX)) ? 0 : lo, a2 = lo & ~3;
    int mt = dft_tiles(n, b0);
    DftShare sh(mt, a.dft.smax);
    // what the update needs, loaded ahead of the transform
    const zd r = a.coef[b];
    const int tA = a.rtab && hasA ? a.rtab_idx[f * a.R + b - 1] : -1, tB = a.rtab && hasB ? a.rtab_idx[f * a.R + b] : -1;
    double xs[TPW][2];
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = b0 + 16 * (sh.first + q * W) + (lane & 15);
        xs[q][0] = a.X[j <= H ? j : H];
        xs[q][1] = a.X[j > 0 && j <= H ? n - j : 0];
    }
    dbl4 e[TPW], o[TPW];
    dft_stage<TPW>(P, part, n, 0, b0, mt, sh, a.dft.tab, e, o);
    // boundary update (src/boost_fractor_recurprop.jl:90-119)
    const zd omr = cmk<double>(1.0 - r.re, -r.im), opr = cmk<double>(1.0 + r.re, r.im), mr = cmk<double>(-r.re, -r.im);
    double vmax = 0.0;
    auto update = [&](int x, double xx, zd& A, zd& B) {
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
        if (fwd && !in_aperture(xx, yy, a.R2)) A = B = cmk<double>(0, 0);  // next bounce's aperture
    };
    if (sh.own(mt) && oky)
#pragma unroll
        for (int q = 0; q < TPW; q++) {
            const int j = b0 + 16 * (sh.first + q * W) + (lane & 15);
            if (sh.first + q * W >= mt || j > H) continue;
            const bool pr = dft_paired(n, j);
            zd A = dft_out(e[q], o[q], 0), B = dft_out(e[q], o[q], 1);
            zd mA = dft_mirror(e[q], o[q], 0), mB = dft_mirror(e[q], o[q], 1);
            update(j, xs[q][0], A, B);
            if (pr)
                update(n - j, xs[q][1], mA, mB);
            else
                mA = mB = cmk<double>(0, 0);
            if (j >= lo) {
                dft_fold<false>(P, j - a2, lane >> 4, A, mA);
                dft_fold<false>(P, j - a2, 4 + (lane >> 4), B, mB);
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
    dft_zero_rows(P, 0, lo - a2);
    dft_zero_rows(P, H + 1 - a2, dft_rows(n, a2));
    mt = dft_tiles(n, 0);
    sh = DftShare(mt, a.dft.smax);
    dft_stage<TPW>(P, part, n, a2, 0, mt, sh, a.dft.tab, e, o);
    if (!sh.own(mt) || !oky) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = 16 * (sh.first + q * W) + (lane & 15);
        if (sh.first + q * W >= mt || j > H) continue;
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
template <typename T>
struct ChPairDftArgs : ChPairArgs<T> {
    int n;
};

template <typename T, int TPW>
__global__ void __launch_bounds__(1024) k_ch_pair_dft(ChPairDftArgs<T> a) {
    using S = typename Storage<T>::type;
    extern __shared__ double2 dft_smem[];
    const int n = a.n, H = n >> 1;
    double2* P = dft_smem;
    double2* part = P + dft_rows(n, 0) * DFT_LDP;
    const int en = blockIdx.y;
    const FieldDesc d0 = a.fd[2 * en], d1 = a.fd[2 * en + 1];
    if (a.active && !a.active[d0.group]) return;  // uniform over the block
    const size_t K = (size_t)n * a.ny;
    const int y0 = a.ylo + blockIdx.x * 4;
    cplx<S>* F0 = a.F + d0.off;
    cplx<S>* F1 = a.F + d1.off;
    const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int c = wave; c < DFT_LINES; c += W) {
        const int yl = y0 + (c & 3);
        dft_load_line<true>(P, n, 0, c, yl < a.yhi ? (c < 4 ? F0 : F1) + (size_t)yl * n : nullptr,
                            [](int, zd v) { return v; });
    }
    const int y = y0 + (lane >> 4);
    const bool oky = y < a.yhi;
    const double yy = a.Y[oky ? y : 0];
    const bool xout = a.xout != 0;
    const int lo = xout ? a.dft.lo : 0, a2 = lo & ~3;  // the mask of the next transform keeps the folded indices >= lo
    int mt = dft_tiles(n, lo);
    DftShare sh(mt, a.dft.smax);
    // what the update needs, loaded ahead of the transform
    const zd* cf = a.coef + 4 * (d0.pad >> FD_PAIR_SHIFT);
    const zd rl = cf[0], tr = cf[1], rr = cf[2], tl = cf[3];
    double xs[TPW][2];
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = lo + 16 * (sh.first + q * W) + (lane & 15);
        xs[q][0] = a.X[j <= H ? j : H];
        xs[q][1] = a.X[j > 0 && j <= H ? n - j : 0];
    }
    dbl4 e[TPW], o[TPW];
    dft_stage<TPW>(P, part, n, 0, lo, mt, sh, a.dft.tab, e, o);
    const int t0 = a.rtab ? d0.rtab : -1, t1 = a.rtab ? d1.rtab : -1;
    // k_ch_pair: Fn = c rl + tr a, Fi = a rr + tl c (a: field i, c: field i+1), rounded as they are stored
    auto update = [&](int x, double xx, zd& A, zd& B) {
        const size_t p = (size_t)y * n + x;
        if (t0 >= 0) A = cmul(A, ccast<double>(a.rtab[(size_t)t0 * K + p]));
        if (t1 >= 0) B = cmul(B, ccast<double>(a.rtab[(size_t)t1 * K + p]));
        A = ccast<double>(ccast<S>(A));
        B = ccast<double>(ccast<S>(B));
        const zd nA = cadd(cmul(A, rr), cmul(tl, B)), nB = cadd(cmul(B, rl), cmul(tr, A));
        A = ccast<double>(ccast<S>(nA));
        B = ccast<double>(ccast<S>(nB));
        if (xout && !in_aperture(xx, yy, a.R2)) A = B = cmk<double>(0, 0);
    };
    if (sh.own(mt) && oky)
#pragma unroll
        for (int q = 0; q < TPW; q++) {
            const int j = lo + 16 * (sh.first + q * W) + (lane & 15);
            if (sh.first + q * W >= mt || j > H) continue;
            const bool pr = dft_paired(n, j);
            zd A = dft_out(e[q], o[q], 0), B = dft_out(e[q], o[q], 1);
            zd mA = dft_mirror(e[q], o[q], 0), mB = dft_mirror(e[q], o[q], 1);
            update(j, xs[q][0], A, B);
            if (pr)
                update(n - j, xs[q][1], mA, mB);
            else
                mA = mB = cmk<double>(0, 0);
            if (xout) {
                dft_fold<false>(P, j - a2, lane >> 4, A, mA);
                dft_fold<false>(P, j - a2, 4 + (lane >> 4), B, mB);
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
    dft_zero_rows(P, 0, lo - a2);
    dft_zero_rows(P, H + 1 - a2, dft_rows(n, a2));
    mt = dft_tiles(n, 0);
    sh = DftShare(mt, a.dft.smax);
    dft_stage<TPW>(P, part, n, a2, 0, mt, sh, a.dft.tab, e, o);
    if (!sh.own(mt) || !oky) return;
#pragma unroll
    for (int q = 0; q < TPW; q++) {
        const int j = 16 * (sh.first + q * W) + (lane & 15);
        if (sh.first + q * W >= mt || j > H) continue;
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
        const size_t planes = sizeof(double2) * DFT_LDP * (size_t)dft_rows(n, 0);
        const size_t part = sizeof(double2) * DFT_PART * (size_t)(waves - 1);
        const bool share = planes + part <= 152 * 1024;
        smax = share ? 4 : 1;
        smem = planes + (share ? part : 0);
    }
};
#define BF_DFT_GO(grid, sh, s, arg, ...)                                                          \
    do {                                                                                          \
        allow_lds((const void*)__VA_ARGS__, (sh).smem);                                           \
        hipLaunchKernelGGL((__VA_ARGS__), grid, dim3(64 * (sh).waves), (sh).smem, s, arg);        \
        BF_CHECK_LAUNCH();                                                                        \
    } while (0)

template <typename T>
void launch_rows_dft(RowArgs<T> a, hipStream_t s) {
    const DftShape sh(a.nx);
    a.dft.smax = sh.smax;
    const long nlines = (long)a.nf * (a.yhi > a.ylo ? a.yhi - a.ylo : a.ny);
    if (nlines > 0x7fffffffL - DFT_LINES) throw Error(BF_ERR_UNSUPPORTED, "too many lines in one row pass");
    const dim3 grid((unsigned)((nlines + DFT_LINES - 1) / DFT_LINES));
    if (sh.tpw == 1)
        BF_DFT_GO(grid, sh, s, a, k_rows_dft<T, 1>);
    else
        BF_DFT_GO(grid, sh, s, a, k_rows_dft<T, 2>);
}
template <typename T>
void launch_cols_dft(ColArgs<T> a, hipStream_t s) {
    const DftShape sh(a.ny);
    a.dft.smax = sh.smax;
    constexpr uint32_t PROP = CF_FWD | CF_KMID | CF_INV;
    const dim3 grid((a.nx + DFT_LINES - 1) / DFT_LINES, a.nf);
    if (a.flags == PROP && a.ktab) {
        if (sh.tpw == 1)
            BF_DFT_GO(grid, sh, s, a, k_cols_dft<T, 1, PROP>);
        else
            BF_DFT_GO(grid, sh, s, a, k_cols_dft<T, 2, PROP>);
    } else {
        if (sh.tpw == 1)
            BF_DFT_GO(grid, sh, s, a, k_cols_dft<T, 1, 0>);
        else
            BF_DFT_GO(grid, sh, s, a, k_cols_dft<T, 2, 0>);
    }
}
template <typename T>
void launch_dancer_rows_dft(DancerRowArgs<T> a, int fb, hipStream_t s) {
    const DftShape sh(a.nx);
    a.dft.smax = sh.smax;
    const unsigned nblk = dancer_tiles(a, 4);
    if (sh.tpw == 1)
        BF_DFT_GO(dim3(nblk, fb), sh, s, a, k_dancer_rows_dft<T, 1>);
    else
        BF_DFT_GO(dim3(nblk, fb), sh, s, a, k_dancer_rows_dft<T, 2>);
}
template <typename T>
void launch_ch_pair_dft(ChPairArgs<T> a, int nx, int entries, hipStream_t s) {
    if (!a.dft.tab) throw std::runtime_error("the pair step's row transforms have no table");
    const DftShape sh(nx);
    a.dft.smax = sh.smax;
    ChPairDftArgs<T> b;
    static_cast<ChPairArgs<T>&>(b) = a;
    b.n = nx;
    const dim3 grid((a.yhi - a.ylo + 3) / 4, entries);
    if (sh.tpw == 1)
        BF_DFT_GO(grid, sh, s, b, k_ch_pair_dft<T, 1>);
    else
        BF_DFT_GO(grid, sh, s, b, k_ch_pair_dft<T, 2>);
}
#define BF_DFT_INSTANCES(T)                                                     \
    template void launch_rows_dft<T>(RowArgs<T>, hipStream_t);                  \
    template void launch_cols_dft<T>(ColArgs<T>, hipStream_t);                  \
    template void launch_dancer_rows_dft<T>(DancerRowArgs<T>, int, hipStream_t); \
    template void launch_ch_pair_dft<T>(ChPairArgs<T>, int, int, hipStream_t);
BF_DFT_INSTANCES(double)
BF_DFT_INSTANCES(float)

// (cos, sin)(2 pi a b / n) for the matrix-core line transforms, a < dft_tab_rows(n), b < dft_ld(n)
__global__ void k_dft_table(double2* out, int n, int ld, int rows) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ld * rows; i += gridDim.x * blockDim.x) {
        const int m = (int)(((long)(i / ld) * (i % ld)) % n);
        double s, c;
        sincospi(2.0 * (double)m / (double)n, &s, &c);
        out[i] = make_double2(c, s);
    }
}
// The context keeps the tables of the last lengths used (at most 4.7 MB each, n = 1023); an
// engine holds its own reference, so a table dropped here lives as long as a plan that reads it.
std::shared_ptr<DevBuf> dft_table(bf_ctx* ctx, int n) {
    auto& cache = ctx->dft_tables;
    for (size_t q = 0; q < cache.size(); q++)
        if (cache[q].first == n) {
            std::rotate(cache.begin() + q, cache.begin() + q + 1, cache.end());
            return cache.back().second;
        }
    const int ld = dft_ld(n), rows = dft_tab_rows(n);
    auto b = std::make_shared<DevBuf>(sizeof(double2) * (size_t)ld * rows);
    hipLaunchKernelGGL(k_dft_table, dim3((ld * rows + 255) / 256), dim3(256), 0, ctx->stream, b->as<double2>(), n, ld,
                       rows);
    BF_CHECK_LAUNCH();
    if (cache.size() >= 8) cache.erase(cache.begin());
    cache.emplace_back(n, b);
    return b;
}

}  // namespace bf
