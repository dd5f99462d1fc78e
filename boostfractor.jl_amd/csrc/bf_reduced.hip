// bf_reduced.hip -- kernels of the bounce solvers' propagation on the aperture's
// window (bf_reduced.h).
#include "bf_reduced.h"
#include "bf_fftmix.h"

#include <algorithm>

namespace bf {

// The two sides of a transform exchange through LDS in FP64 whatever the storage: rounding
// the exchanges of complex64 fields too is 5% faster (20 disks, 256^2: 45.0 against 47.2 ms
// for 20 frequencies x 201 bounces) but raises the error against FP64.
// columns per block of the column pass: 128 or 256 bytes of a row, at most 41 KB of LDS
template <int R>
struct RdCol {
    static constexpr int C = R <= 10 ? 16 : 8;
    static constexpr int NT = C * (R > 16 ? R : 16);
    // 128 VGPRs (a few below what the compiler takes on its own) let a second block on the CU
    static constexpr int WPE = R <= 10 ? 4 : 3;
};
// rows per block of the row pass (two lines each): at most 44 KB of LDS
template <int R>
struct RdRow {
    static constexpr int L = R <= 6 ? 8 : 4;
    static constexpr int NA = 32 * L, NB = 2 * L * R, NT = ((NA > NB ? NA : NB) + 63) / 64 * 64;
    static constexpr int LD = R * 17;  // [k1][17]: the radix-16 side writes, the radix-R side reads without conflicts
};

// the 16 wavenumbers k1 + R q of a stored line
template <int R>
__device__ __forceinline__ void rd_load(const cplx<float>* f, int k1, cplx<float> (&v)[16]) {
#pragma unroll
    for (int q = 0; q < 16; q += 2) {
        const float4 w = *reinterpret_cast<const float4*>(f + rd_pos<true>(R, k1, q));
        v[q] = cmk<float>(w.x, w.y);
        v[q + 1] = cmk<float>(w.z, w.w);
    }
}
template <int R>
__device__ __forceinline__ void rd_load(const cplx<double>* f, int k1, cplx<double> (&v)[16]) {
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = f[rd_pos<false>(R, k1, q)];
}
template <int R>
__device__ __forceinline__ void rd_store(cplx<float>* f, int k1, const zd (&v)[16]) {
#pragma unroll
    for (int q = 0; q < 16; q += 2)
        *reinterpret_cast<float4*>(f + rd_pos<true>(R, k1, q)) =
            make_float4((float)v[q].re, (float)v[q].im, (float)v[q + 1].re, (float)v[q + 1].im);
}
template <int R>
__device__ __forceinline__ void rd_store(cplx<double>* f, int k1, const zd (&v)[16]) {
#pragma unroll
    for (int q = 0; q < 16; q++) f[rd_pos<false>(R, k1, q)] = v[q];
}

// Column pass: transform along y, times the table, and back, window rows in and out.
// Threads (t, column) for the samples, (k1, column) for the wavenumbers; neighbouring
// lanes are neighbouring columns, in HBM and in LDS.  Bound by the traffic behind L2: 10 frequencies
// of 20 disks on 256^2 (R = 10) move 464 MB, 323 of them the fields, in 74 us, 6.3 TB/s, with FP64
// issue at 0.41 and LDS at 0.25 of the time (the row pass: 322 MB in 54 us, FP64 issue 0.36).  Both
// passes, 20 disks on 256^2 (20 frequencies x 201 bounces), take 53 ms against 82 on the whole grid,
// 512^2 (4 x 101) 24 against 52; 3 disks on 101^2 (16 x 201) 3.7 against 9.2.
template <typename S, int R>
__global__ void __launch_bounds__((RdCol<R>::NT)) __attribute__((amdgpu_waves_per_eu(RdCol<R>::WPE))) k_rd_cols(RdColArgs<S> a) {
    constexpr int C = RdCol<R>::C, H = rd_half(R);
    constexpr uint32_t SZ = sizeof(cplx<S>);
    __shared__ zd sm[16 * R * C];
    const FieldDesc d = a.fd[blockIdx.y];
    const int c = threadIdx.x % C, t = threadIdx.x / C, x = blockIdx.x * C + c;
    const int Mx = 16 * a.Rx;
    const bool ok = x < Mx;
    const uint32_t rowb = (uint32_t)Mx * SZ;
    const auto rf = buf_rsrc(a.F + d.off, (uint32_t)a.by * rowb);  // rows past the window read as zero
    const uint32_t o0 = ok && t < 16 ? (uint32_t)t * rowb + (uint32_t)x * SZ : BUF_OOB;
    // byte offset of sample t + 16 m beyond o0, never past the field's end: what lies beyond the resource's
    // length less this offset is out of range, and that difference is not to be negative
    auto rows16 = [&](int m) { return (uint32_t)min(16 * m, a.by) * rowb; };
    const zd* tw = a.tw + (t < 16 ? t : 0);
    zd* s = sm + c;
    if (t < 16) {
        cplx<S> raw[H];
#pragma unroll
        for (int m = 0; m < H; m++) raw[m] = buf_load<S>(rf, o0, rows16(m));
        if (d.rtab >= 0 && ok) {  // uniform but for the last columns
            zd* q = a.sum + ((size_t)d.rtab * a.by + t) * Mx + x;
#pragma unroll
            for (int m = 0; m < H; m++)
                if (t + 16 * m < a.by) {
                    zd* p = q + (size_t)(16 * m) * Mx;
                    *p = cadd(*p, ccast<double>(raw[m]));
                }
        }
        if (!(d.pad & RD_SUM_ONLY)) {
            zd v[R];
#pragma unroll
            for (int m = 0; m < H; m++) v[m] = ccast<double>(raw[m]);
            dft_in<R, false>(v);
            s[(t * R) * C] = v[0];
#pragma unroll
            for (int k1 = 1; k1 < R; k1++) s[(t * R + k1) * C] = cmul(v[k1], tw[16 * k1]);
        }
    }
    if (d.pad & RD_SUM_ONLY) return;  // uniform over the block
    // table entries of this thread's wavenumbers t + R q: rows past the middle are the mirror
    // rows (16 - q) R - t of a quarter table, and the column's wavenumber its mirror
    const int kx = rd_wavenumber<sizeof(S) == 4>(a.Rx, x), W = a.quarter ? Mx / 2 + 1 : Mx;
    const uint32_t krow = (uint32_t)W * (uint32_t)sizeof(zd), kb = (uint32_t)(a.quarter && 2 * kx > Mx ? Mx - kx : kx) * (uint32_t)sizeof(zd);
    const uint32_t KT = (a.quarter ? 8u * R + 1u : 16u * R) * krow;
    const auto rk = buf_rsrc(reinterpret_cast<const char*>(a.tab) + (size_t)d.ktab * KT, KT);
    const bool onk = ok && t < R;
    const uint32_t klo = onk ? kb + (uint32_t)t * krow : BUF_OOB, khi = onk && a.quarter ? kb + (uint32_t)(R - t) * krow : klo;
    constexpr int KCH = 8;
    zd k[KCH];
    auto fetch = [&](int q0) {
#pragma unroll
        for (int q = 0; q < KCH; q++) {
            const uint32_t r = q0 == 0 || !a.quarter ? (uint32_t)(R * (q0 + q)) : (uint32_t)(R * (15 - q0 - q));
            k[q] = buf_load<double>(rk, q0 == 0 ? klo : khi, r * krow);
        }
    };
    fetch(0);
    __syncthreads();
    if (t < R) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = s[(q * R + t) * C];
        dft_reg<double, 16, false>(v);
#pragma unroll
        for (int q = 0; q < KCH; q++) v[q] = cmul(v[q], k[q]);
        fetch(KCH);
#pragma unroll
        for (int q = 0; q < KCH; q++) v[KCH + q] = cmul(v[KCH + q], k[q]);
        dft_reg<double, 16, true>(v);
#pragma unroll
        for (int q = 0; q < 16; q++) s[(q * R + t) * C] = v[q];
    }
    __syncthreads();
    if (t < 16) {
        zd v[R];
        v[0] = s[(t * R) * C];
#pragma unroll
        for (int k1 = 1; k1 < R; k1++) v[k1] = cmulc(s[(t * R + k1) * C], tw[16 * k1]);
        dft_out_half<R, true>(v);
#pragma unroll
        for (int m = 0; m < H; m++)
            buf_store<S>(rf, o0, ccast<S>(v[m]), rows16(m));
    }
}

// Row pass: both fields of a boundary back along x, tilt/surface, the 2 x 2 update, the
// aperture, and along x again.  Threads (row, field, t) hold the samples of one field's
// row; the other field's are 16 lanes away.  (k1, line) loads and stores the wavenumbers.
template <typename S, int R>
__global__ void __launch_bounds__((RdRow<R>::NT)) k_rd_pairs(RdPairArgs<S> a) {
    using P = RdRow<R>;
    constexpr int L = P::L, LD = P::LD, H = rd_half(R), Mx = 16 * R;
    __shared__ zd sm[2 * L * LD];
    const RdPair e = a.pairs[blockIdx.y];
    const int y0 = blockIdx.x * L, tid = threadIdx.x;
    if (e.flags & RP_ZERO0) {  // uniform over the block
        for (int q = tid; q < L * Mx; q += P::NT)
            if (y0 + q / Mx < a.by) a.F[e.off0 + (int64_t)y0 * Mx + q] = cmk<S>(0, 0);
        return;
    }
    // wavenumber side
    const int k1 = tid % R, line = tid / R, fb = line & 1, yb = y0 + (line >> 1);
    const bool onb = tid < P::NB && yb < a.by;
    cplx<S>* f = a.F + (fb == 0 ? e.off0 : e.off1) + (int64_t)(onb ? yb : 0) * Mx;
    zd* sb = sm + line * LD + k1 * 17;
    if (tid < P::NB) {
        if (onb && (e.flags & (fb == 0 ? RP_LOAD0 : RP_LOAD1))) {
            cplx<S> raw[16];
            rd_load<R>(f, k1, raw);
            zd v[16];
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = ccast<double>(raw[q]);
            dft_reg<double, 16, true>(v);
#pragma unroll
            for (int q = 0; q < 16; q++) sb[q] = v[q];
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++) sb[q] = cmk<double>(0, 0);
        }
    }
    // sample side: what the update needs, ahead of the barrier
    const int t = tid % 16, fa = (tid / 16) & 1, row = tid / 32, y = y0 + row;
    const uint32_t keep = tid < P::NA && y < a.by ? a.keep[y * 16 + t] : 0u;
    const zd* cf = a.coef + 4 * (int64_t)e.coef;
    const zd own = fa == 0 ? cf[0] : cf[3], other = fa == 0 ? cf[1] : cf[2];
    const int rt = fa == 0 ? e.rt0 : e.rt1;
    __syncthreads();
    if (tid < P::NA) {  // whole waves
        const zd* tw = a.tw + t;
        zd* s = sm + (2 * row + fa) * LD + t;
        zd u[H];
        {
            zd v[R];
            v[0] = s[0];
#pragma unroll
            for (int q = 1; q < R; q++) v[q] = cmulc(s[17 * q], tw[16 * q]);
            dft_out_half<R, true>(v);
#pragma unroll
            for (int m = 0; m < H; m++) u[m] = v[m];
        }
        if (rt >= 0) {
            const zd* tp = a.rtab + (size_t)rt * a.K + (size_t)(a.y0 + y) * a.nx + a.x0 + t;
#pragma unroll
            for (int m = 0; m < H; m++)
                if ((keep >> m) & 1u) u[m] = cmul(u[m], tp[16 * m]);
        }
#pragma unroll
        for (int m = 0; m < H; m++) {
            const zd w = cmk<double>(__shfl_xor(u[m].re, 16), __shfl_xor(u[m].im, 16));
            const zd n = cmac(cmul(u[m], own), other, w);
            u[m] = (keep >> m) & 1u ? n : cmk<double>(0, 0);
        }
        zd v[R];
#pragma unroll
        for (int m = 0; m < H; m++) v[m] = u[m];
        dft_in<R, false>(v);
        s[0] = v[0];
#pragma unroll
        for (int q = 1; q < R; q++) s[17 * q] = cmul(v[q], tw[16 * q]);
    }
    __syncthreads();
    if (onb && (e.flags & (fb == 0 ? RP_STORE0 : RP_STORE1 | RP_ADD1))) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = sb[q];
        dft_reg<double, 16, false>(v);
        if (fb == 1 && (e.flags & RP_ADD1)) {
            cplx<S> raw[16];
            rd_load<R>(f, k1, raw);
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = cadd(ccast<double>(raw[q]), v[q]);
        }
        rd_store<R>(f, k1, v);
    }
}

// lines per block of the two kernels below
template <int R>
struct RdLine {
    static constexpr int N = R > 10 ? 8 : 16, NT = N * (R > 16 ? R : 16), LD = R * 17;
};

template <typename S, int R>
__global__ void __launch_bounds__((RdLine<R>::NT)) k_rd_init(RdInitArgs<S> a) {
    constexpr int LD = RdLine<R>::LD, H = rd_half(R), Mx = 16 * R, LINES = RdLine<R>::N;
    __shared__ zd sm[LINES * LD];
    const FieldDesc d = a.fd[blockIdx.y];
    const int y0 = blockIdx.x * LINES, tid = threadIdx.x;
    if (a.add && d.ktab < 0) return;  // uniform over the block
    if (tid < 16 * LINES) {
        const int t = tid % 16, row = tid / 16, y = y0 + row;
        const uint32_t keep = y < a.by && d.ktab >= 0 ? a.keep[y * 16 + t] : 0u;
        zd v[R];
#pragma unroll
        for (int m = 0; m < H; m++) {
            v[m] = cmk<double>(0, 0);
            if ((keep >> m) & 1u) {
                double sn, cs;
                sincospi(a.ex * (double)(t + 16 * m) + a.ey * (double)y, &sn, &cs);
                v[m] = cmul(cmk<double>(cs, sn), a.amp ? a.amp[d.ktab]
                                                       : a.src[(size_t)d.ktab * a.K + (size_t)(a.y0 + y) * a.nx + a.x0 + t + 16 * m]);
            }
        }
        dft_in<R, false>(v);
        zd* s = sm + row * LD + t;
        s[0] = v[0];
#pragma unroll
        for (int q = 1; q < R; q++) s[17 * q] = cmul(v[q], a.tw[16 * q + t]);
    }
    __syncthreads();
    const int k1 = tid % R, line = tid / R, y = y0 + line;
    if (line < LINES && y < a.by) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = sm[line * LD + k1 * 17 + q];
        dft_reg<double, 16, false>(v);
        cplx<S>* f = a.F + d.off + (int64_t)y * Mx;
        if (a.add) {
            cplx<S> raw[16];
            rd_load<R>(f, k1, raw);
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = cadd(ccast<double>(raw[q]), v[q]);
        }
        rd_store<R>(f, k1, v);
    }
}

template <int R, bool PAIR>
__global__ void __launch_bounds__((RdLine<R>::NT)) k_rd_final(RdFinalArgs a) {
    constexpr int LD = RdLine<R>::LD, H = rd_half(R), Mx = 16 * R, LINES = RdLine<R>::N;
    __shared__ zd sm[LINES * LD];
    const int y0 = blockIdx.x * LINES, tid = threadIdx.x;
    const int k1 = tid % R, line = tid / R;
    if (line < LINES) {
        zd v[16];
        const bool on = y0 + line < a.by;
        const zd* f = a.sum + ((size_t)blockIdx.y * a.by + (on ? y0 + line : 0)) * Mx;
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = on ? f[rd_pos<PAIR>(R, k1, q)] : cmk<double>(0, 0);
        dft_reg<double, 16, true>(v);
#pragma unroll
        for (int q = 0; q < 16; q++) sm[line * LD + k1 * 17 + q] = v[q];
    }
    __syncthreads();
    const int t = tid % 16, row = tid / 16, y = y0 + row;
    if (row < LINES && y < a.by) {
        const zd* s = sm + row * LD + t;
        zd v[R];
        v[0] = s[0];
#pragma unroll
        for (int q = 1; q < R; q++) v[q] = cmulc(s[17 * q], a.tw[16 * q + t]);
        dft_out_half<R, true>(v);
        zd* o = a.out + (size_t)blockIdx.y * a.K + (size_t)(a.y0 + y) * a.nx + a.x0 + t;
        const double sc = 1.0 / (double)Mx;
#pragma unroll
        for (int m = 0; m < H; m++)
            if (t + 16 * m < a.bx) {
                double sn, cs;
                sincospi(a.ex * (double)(t + 16 * m) + a.ey * (double)y, &sn, &cs);
                o[16 * m] = cmul(cmk<double>(sc * cs, -sc * sn), v[m]);
            }
    }
}

__global__ void k_rd_crop(const zd* __restrict__ h, int nx, int ny, int by, int bx, int My, int Mx,
                          double ey, double ex, zd* out) {
    const double sc = 1.0 / ((double)My * (double)Mx);
    const size_t K = (size_t)nx * ny, KM = (size_t)My * Mx;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < KM; i += (size_t)gridDim.x * blockDim.x) {
        const int my = (int)(i / Mx), mx = (int)(i % Mx);
        const int dy = my < by ? my : my - My, dx = mx < bx ? mx : mx - Mx;
        zd v = cmk<double>(0, 0);
        if (dy > -by && dx > -bx) {
            const int sy = ((dy % ny) + ny) % ny, sx = ((dx % nx) + nx) % nx;
            const zd u = h[blockIdx.y * K + (size_t)sy * nx + sx];
            double sn, cs;
            sincospi(ey * (double)dy + ex * (double)dx, &sn, &cs);
            v = cmul(cmk<double>(sc * cs, sc * sn), u);
        }
        out[blockIdx.y * KM + i] = v;
    }
}

__global__ void k_rd_quarter(const zd* __restrict__ full, int My, int Mx, zd* out) {
    const int W = Mx / 2 + 1, n = W * (My / 2 + 1);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        out[(size_t)blockIdx.y * n + i] = full[((size_t)blockIdx.y * My + i / W) * Mx + i % W];
}

__global__ void k_rd_twiddles(zd* out, int R) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 16 * R) return;
    double s, c;
    sincospi(2.0 * (double)((i / 16) * (i % 16)) / (double)(16 * R), &s, &c);
    out[i] = cmk<double>(c, -s);
}

void rd_crop(const RdShape& sh, const zd* h, int nx, int ny, int ntab, zd* out, hipStream_t s) {
    const unsigned gx = (unsigned)std::min<size_t>((sh.points() + 255) / 256, 1024);
    hipLaunchKernelGGL(k_rd_crop, dim3(gx, ntab), dim3(256), 0, s, h, nx, ny, sh.by, sh.bx, sh.My(), sh.Mx(),
                       sh.ey, sh.ex, out);
    BF_CHECK_LAUNCH();
}
void rd_quarter(const RdShape& sh, const zd* full, int ntab, zd* out, hipStream_t s) {
    hipLaunchKernelGGL(k_rd_quarter, dim3((unsigned)((sh.table() + 255) / 256), ntab), dim3(256), 0, s, full, sh.My(),
                       sh.Mx(), out);
    BF_CHECK_LAUNCH();
}
void rd_twiddles(int R, zd* out, hipStream_t s) {
    hipLaunchKernelGGL(k_rd_twiddles, dim3((16 * R + 255) / 256), dim3(256), 0, s, out, R);
    BF_CHECK_LAUNCH();
}

#define RD_EACH(X, R_)                                                                                  \
    switch (R_) {                                                                                       \
        case 4: X(4); break;                                                                            \
        case 5: X(5); break;                                                                            \
        case 6: X(6); break;                                                                            \
        case 8: X(8); break;                                                                            \
        case 10: X(10); break;                                                                          \
        case 12: X(12); break;                                                                          \
        case 16: X(16); break;                                                                          \
        case 20: X(20); break;                                                                          \
        default: throw Error(BF_ERR_UNSUPPORTED, "no reduced line of " + std::to_string(16 * (R_)) + " points"); \
    }

template <typename S>
void rd_cols(const RdShape& sh, const RdColArgs<S>& a, int nf, hipStream_t s) {
    if (nf <= 0) return;
#define GO(R)                                                                                             \
    hipLaunchKernelGGL((k_rd_cols<S, R>), dim3((sh.Mx() + RdCol<R>::C - 1) / RdCol<R>::C, nf),            \
                       dim3(RdCol<R>::NT), 0, s, a)
    RD_EACH(GO, sh.Ry)
#undef GO
    BF_CHECK_LAUNCH();
}
template <typename S>
void rd_pairs(const RdShape& sh, const RdPairArgs<S>& a, int n, hipStream_t s) {
    if (n <= 0) return;
#define GO(R)                                                                                             \
    hipLaunchKernelGGL((k_rd_pairs<S, R>), dim3((sh.by + RdRow<R>::L - 1) / RdRow<R>::L, n),              \
                       dim3(RdRow<R>::NT), 0, s, a)
    RD_EACH(GO, sh.Rx)
#undef GO
    BF_CHECK_LAUNCH();
}
template <typename S>
void rd_init(const RdShape& sh, const RdInitArgs<S>& a, int nf, hipStream_t s) {
    if (nf <= 0) return;
#define GO(R)                                                                                                   \
    hipLaunchKernelGGL((k_rd_init<S, R>), dim3((sh.by + RdLine<R>::N - 1) / RdLine<R>::N, nf), dim3(RdLine<R>::NT), 0, s, a)
    RD_EACH(GO, sh.Rx)
#undef GO
    BF_CHECK_LAUNCH();
}
void rd_final(const RdShape& sh, const RdFinalArgs& a, int n, bool pair, hipStream_t s) {
    if (n <= 0) return;
#define GO(R)                                                                                                   \
    if (pair)                                                                                                   \
        hipLaunchKernelGGL((k_rd_final<R, true>), dim3((sh.by + RdLine<R>::N - 1) / RdLine<R>::N, n),           \
                           dim3(RdLine<R>::NT), 0, s, a);                                                       \
    else                                                                                                        \
        hipLaunchKernelGGL((k_rd_final<R, false>), dim3((sh.by + RdLine<R>::N - 1) / RdLine<R>::N, n),          \
                           dim3(RdLine<R>::NT), 0, s, a)
    RD_EACH(GO, sh.Rx)
#undef GO
    BF_CHECK_LAUNCH();
}
template void rd_cols<float>(const RdShape&, const RdColArgs<float>&, int, hipStream_t);
template void rd_cols<double>(const RdShape&, const RdColArgs<double>&, int, hipStream_t);
template void rd_pairs<float>(const RdShape&, const RdPairArgs<float>&, int, hipStream_t);
template void rd_pairs<double>(const RdShape&, const RdPairArgs<double>&, int, hipStream_t);
template void rd_init<float>(const RdShape&, const RdInitArgs<float>&, int, hipStream_t);
template void rd_init<double>(const RdShape&, const RdInitArgs<double>&, int, hipStream_t);

}  // namespace bf
