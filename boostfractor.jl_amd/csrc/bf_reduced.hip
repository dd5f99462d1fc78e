// bf_reduced.hip -- kernels of the bounce solvers' propagation on the aperture's
// window (bf_reduced.h).
#include "bf_reduced.h"
#include "bf_fftmix.h"

#include <algorithm>

namespace bf {

// columns per block of the column pass: 41 KB of LDS at R = 10 and 20
template <typename S, int R>
struct RdCol {
    static constexpr int C = (sizeof(S) == 4 ? 32 : 16) / (R > 10 ? 2 : 1);
    static constexpr int NT = C * (R > 16 ? R : 16);
};
// row pairs per block of the row pass (two lines each)
template <typename S, int R>
struct RdRow {
    static constexpr int L = (sizeof(S) == 4 ? 16 : 8) / (R > 10 ? 2 : 1);
    static constexpr int NA = 16 * L, NB = 2 * L * R, NT = ((NA > NB ? NA : NB) + 63) / 64 * 64;
    static constexpr int LD = R * 17;  // [k1][17]: the radix-16 side writes, the radix-R side reads without conflicts
};

// Column pass: transform along y, times the table, and back, window rows in and out.
// Threads (t, column) for the samples, (k1, column) for the wavenumbers; neighbouring
// lanes are neighbouring columns, in HBM and in LDS.  VALU-bound in FP64 arithmetic:
// 630 instructions per lane at R = 10 for 16 (10) lanes a line.
template <typename S, int R>
__global__ void __launch_bounds__((RdCol<S, R>::NT)) k_rd_cols(RdColArgs<S> a) {
    constexpr int C = RdCol<S, R>::C, H = rd_half(R);
    constexpr uint32_t SZ = sizeof(cplx<S>);
    __shared__ cplx<S> sm[16 * R * C];
    const FieldDesc d = a.fd[blockIdx.y];
    const int c = threadIdx.x % C, t = threadIdx.x / C, x = blockIdx.x * C + c;
    const bool ok = x < a.Mx;
    const uint32_t rowb = (uint32_t)a.Mx * SZ;
    const auto rf = buf_rsrc(a.F + d.off, (uint32_t)a.by * rowb);  // rows past the window read as zero
    const uint32_t o0 = ok && t < 16 ? (uint32_t)t * rowb + (uint32_t)x * SZ : BUF_OOB;
    const zd* tw = a.tw + (t < 16 ? t : 0);
    cplx<S>* s = sm + c;
    if (t < 16) {
        cplx<S> raw[H];
#pragma unroll
        for (int m = 0; m < H; m++) raw[m] = buf_load<S>(rf, o0 == BUF_OOB ? BUF_OOB : o0 + (uint32_t)(16 * m) * rowb);
        if (d.rtab >= 0 && ok) {  // uniform but for the last columns
            zd* q = a.sum + ((size_t)d.rtab * a.by + t) * a.Mx + x;
#pragma unroll
            for (int m = 0; m < H; m++)
                if (t + 16 * m < a.by) {
                    zd* p = q + (size_t)(16 * m) * a.Mx;
                    *p = cadd(*p, ccast<double>(raw[m]));
                }
        }
        if (!(d.pad & RD_SUM_ONLY)) {
            zd v[R];
#pragma unroll
            for (int m = 0; m < H; m++) v[m] = ccast<double>(raw[m]);
            dft_in<R, false>(v);
            s[(t * R) * C] = ccast<S>(v[0]);
#pragma unroll
            for (int k1 = 1; k1 < R; k1++) s[(t * R + k1) * C] = ccast<S>(cmul(v[k1], tw[16 * k1]));
        }
    }
    if (d.pad & RD_SUM_ONLY) return;  // uniform over the block
    const uint32_t krow = (uint32_t)a.Mx * (uint32_t)sizeof(zd);
    const auto rk = buf_rsrc(a.tab + (size_t)d.ktab * 16 * R * a.Mx, 16u * R * krow);
    const uint32_t k0 = ok && t < R ? (uint32_t)t * krow + (uint32_t)x * (uint32_t)sizeof(zd) : BUF_OOB;
    constexpr int KCH = 8;
    zd k[KCH];
    auto fetch = [&](int q0) {
#pragma unroll
        for (int q = 0; q < KCH; q++) k[q] = buf_load<double>(rk, k0 == BUF_OOB ? BUF_OOB : k0 + (uint32_t)(R * (q0 + q)) * krow);
    };
    fetch(0);
    __syncthreads();
    if (t < R) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = ccast<double>(s[(q * R + t) * C]);
        dft_reg<double, 16, false>(v);
#pragma unroll
        for (int q = 0; q < KCH; q++) v[q] = cmul(v[q], k[q]);
        fetch(KCH);
#pragma unroll
        for (int q = 0; q < KCH; q++) v[KCH + q] = cmul(v[KCH + q], k[q]);
        dft_reg<double, 16, true>(v);
#pragma unroll
        for (int q = 0; q < 16; q++) s[(q * R + t) * C] = ccast<S>(v[q]);
    }
    __syncthreads();
    if (t < 16) {
        zd v[R];
        v[0] = ccast<double>(s[(t * R) * C]);
#pragma unroll
        for (int k1 = 1; k1 < R; k1++) v[k1] = cmulc(ccast<double>(s[(t * R + k1) * C]), tw[16 * k1]);
        dft_out_half<R, true>(v);
#pragma unroll
        for (int m = 0; m < H; m++)
            buf_store<S>(rf, o0 == BUF_OOB ? BUF_OOB : o0 + (uint32_t)(16 * m) * rowb, ccast<S>(v[m]));
    }
}

// Row pass: both fields of a boundary back along x, tilt/surface, the 2 x 2 update, the
// aperture, and along x again.  Thread (t, row) holds both fields' samples of its row,
// so the update needs no exchange; (k1, line) loads and stores the wavenumbers.
template <typename S, int R>
__global__ void __launch_bounds__((RdRow<S, R>::NT)) k_rd_pairs(RdPairArgs<S> a) {
    using P = RdRow<S, R>;
    constexpr int L = P::L, LD = P::LD, H = rd_half(R), Mx = 16 * R;
    __shared__ cplx<S> sm[2 * L * LD];
    const RdPair e = a.pairs[blockIdx.y];
    const int y0 = blockIdx.x * L, tid = threadIdx.x;
    if (e.flags & RP_ZERO0) {  // uniform over the block
        for (int q = tid; q < L * Mx; q += P::NT)
            if (y0 + q / Mx < a.by) a.F[e.off0 + (int64_t)y0 * Mx + q] = cmk<S>(0, 0);
        return;
    }
    // wavenumber side
    const int k1 = tid % R, line = tid / R, side = line / L, yb = y0 + line % L;
    const bool onb = tid < P::NB && yb < a.by;
    cplx<S>* f = a.F + (side == 0 ? e.off0 : e.off1) + (int64_t)(onb ? yb : 0) * Mx + k1;
    cplx<S>* sb = sm + line * LD + k1 * 17;
    if (tid < P::NB) {
        if (onb && (e.flags & (side == 0 ? RP_LOAD0 : RP_LOAD1))) {
            cplx<S> raw[16];
#pragma unroll
            for (int q = 0; q < 16; q++) raw[q] = f[R * q];
            zd v[16];
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = ccast<double>(raw[q]);
            dft_reg<double, 16, true>(v);
#pragma unroll
            for (int q = 0; q < 16; q++) sb[q] = ccast<S>(v[q]);
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++) sb[q] = cmk<S>(0, 0);
        }
    }
    // sample side: what the update needs, ahead of the barrier
    const int t = tid % 16, row = tid / 16, y = y0 + row;
    const bool ona = tid < P::NA && y < a.by;
    const uint32_t keep = ona ? a.keep[y * 16 + t] : 0u;
    const zd* cf = a.coef + 4 * (int64_t)e.coef;
    const zd c0 = cf[0], c1 = cf[1], c2 = cf[2], c3 = cf[3];
    __syncthreads();
    if (ona) {
        const zd* tw = a.tw + t;
        cplx<S>* s0 = sm + row * LD + t;
        cplx<S>* s1 = s0 + L * LD;
        zd u[H], w[H];
        auto back = [&](const cplx<S>* s, zd (&out)[H]) {
            zd v[R];
            v[0] = ccast<double>(s[0]);
#pragma unroll
            for (int q = 1; q < R; q++) v[q] = cmulc(ccast<double>(s[17 * q]), tw[16 * q]);
            dft_out_half<R, true>(v);
#pragma unroll
            for (int m = 0; m < H; m++) out[m] = v[m];
        };
        back(s0, u);
        back(s1, w);
        if (e.rt0 >= 0 || e.rt1 >= 0) {
            const size_t p = (size_t)(a.y0 + y) * a.nx + a.x0 + t;
#pragma unroll
            for (int m = 0; m < H; m++)
                if ((keep >> m) & 1u) {
                    if (e.rt0 >= 0) u[m] = cmul(u[m], a.rtab[(size_t)e.rt0 * a.K + p + 16 * m]);
                    if (e.rt1 >= 0) w[m] = cmul(w[m], a.rtab[(size_t)e.rt1 * a.K + p + 16 * m]);
                }
        }
#pragma unroll
        for (int m = 0; m < H; m++) {
            const bool in = (keep >> m) & 1u;
            const zd nu = cmac(cmul(u[m], c0), c1, w[m]), nw = cmac(cmul(w[m], c3), c2, u[m]);
            u[m] = in ? nu : cmk<double>(0, 0);
            w[m] = in ? nw : cmk<double>(0, 0);
        }
        auto forth = [&](cplx<S>* s, const zd (&in)[H]) {
            zd v[R];
#pragma unroll
            for (int m = 0; m < H; m++) v[m] = in[m];
            dft_in<R, false>(v);
            s[0] = ccast<S>(v[0]);
#pragma unroll
            for (int q = 1; q < R; q++) s[17 * q] = ccast<S>(cmul(v[q], tw[16 * q]));
        };
        forth(s0, u);
        forth(s1, w);
    }
    __syncthreads();
    if (onb && (e.flags & (side == 0 ? RP_STORE0 : RP_STORE1 | RP_ADD1))) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = ccast<double>(sb[q]);
        dft_reg<double, 16, false>(v);
        if (side == 1 && (e.flags & RP_ADD1)) {
            cplx<S> raw[16];
#pragma unroll
            for (int q = 0; q < 16; q++) raw[q] = f[R * q];
#pragma unroll
            for (int q = 0; q < 16; q++) v[q] = cadd(ccast<double>(raw[q]), v[q]);
        }
#pragma unroll
        for (int q = 0; q < 16; q++) f[R * q] = ccast<S>(v[q]);
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
    __shared__ cplx<S> sm[LINES * LD];
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
            if ((keep >> m) & 1u)
                v[m] = a.amp ? a.amp[d.ktab] : a.src[(size_t)d.ktab * a.K + (size_t)(a.y0 + y) * a.nx + a.x0 + t + 16 * m];
        }
        dft_in<R, false>(v);
        cplx<S>* s = sm + row * LD + t;
        s[0] = ccast<S>(v[0]);
#pragma unroll
        for (int q = 1; q < R; q++) s[17 * q] = ccast<S>(cmul(v[q], a.tw[16 * q + t]));
    }
    __syncthreads();
    const int k1 = tid % R, line = tid / R, y = y0 + line;
    if (line < LINES && y < a.by) {
        zd v[16];
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = ccast<double>(sm[line * LD + k1 * 17 + q]);
        dft_reg<double, 16, false>(v);
        cplx<S>* f = a.F + d.off + (int64_t)y * Mx + k1;
#pragma unroll
        for (int q = 0; q < 16; q++) f[R * q] = a.add ? ccast<S>(cadd(ccast<double>(f[R * q]), v[q])) : ccast<S>(v[q]);
    }
}

template <int R>
__global__ void __launch_bounds__((RdLine<R>::NT)) k_rd_final(RdFinalArgs a) {
    constexpr int LD = RdLine<R>::LD, H = rd_half(R), Mx = 16 * R, LINES = RdLine<R>::N;
    __shared__ zd sm[LINES * LD];
    const int y0 = blockIdx.x * LINES, tid = threadIdx.x;
    const int k1 = tid % R, line = tid / R;
    if (line < LINES) {
        zd v[16];
        const bool on = y0 + line < a.by;
        const zd* f = a.sum + ((size_t)blockIdx.y * a.by + (on ? y0 + line : 0)) * Mx + k1;
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = on ? f[R * q] : cmk<double>(0, 0);
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
            if (t + 16 * m < a.bx) o[16 * m] = cmk<double>(v[m].re * sc, v[m].im * sc);
    }
}

__global__ void k_rd_crop(const zd* __restrict__ h, int nx, int ny, int by, int bx, int My, int Mx, zd* out) {
    const double sc = 1.0 / ((double)My * (double)Mx);
    const size_t K = (size_t)nx * ny, KM = (size_t)My * Mx;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < KM; i += (size_t)gridDim.x * blockDim.x) {
        const int my = (int)(i / Mx), mx = (int)(i % Mx);
        const int dy = my < by ? my : my - My, dx = mx < bx ? mx : mx - Mx;
        zd v = cmk<double>(0, 0);
        if (dy > -by && dx > -bx) {
            const int sy = ((dy % ny) + ny) % ny, sx = ((dx % nx) + nx) % nx;
            const zd u = h[blockIdx.y * K + (size_t)sy * nx + sx];
            v = cmk<double>(u.re * sc, u.im * sc);
        }
        out[blockIdx.y * KM + i] = v;
    }
}

__global__ void k_rd_twiddles(zd* out, int R) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 16 * R) return;
    double s, c;
    sincospi(2.0 * (double)((i / 16) * (i % 16)) / (double)(16 * R), &s, &c);
    out[i] = cmk<double>(c, -s);
}

void rd_crop(const RdShape& sh, const zd* h, int nx, int ny, int ntab, zd* out, hipStream_t s) {
    const unsigned gx = (unsigned)std::min<size_t>((sh.table() + 255) / 256, 1024);
    hipLaunchKernelGGL(k_rd_crop, dim3(gx, ntab), dim3(256), 0, s, h, nx, ny, sh.by, sh.bx, sh.My(), sh.Mx(), out);
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
#define GO(R)                                                                                                   \
    hipLaunchKernelGGL((k_rd_cols<S, R>), dim3((sh.Mx() + RdCol<S, R>::C - 1) / RdCol<S, R>::C, nf),            \
                       dim3(RdCol<S, R>::NT), 0, s, a)
    RD_EACH(GO, sh.Ry)
#undef GO
    BF_CHECK_LAUNCH();
}
template <typename S>
void rd_pairs(const RdShape& sh, const RdPairArgs<S>& a, int n, hipStream_t s) {
    if (n <= 0) return;
#define GO(R)                                                                                                   \
    hipLaunchKernelGGL((k_rd_pairs<S, R>), dim3((sh.by + RdRow<S, R>::L - 1) / RdRow<S, R>::L, n),              \
                       dim3(RdRow<S, R>::NT), 0, s, a)
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
void rd_final(const RdShape& sh, const RdFinalArgs& a, int n, hipStream_t s) {
    if (n <= 0) return;
#define GO(R) \
    hipLaunchKernelGGL((k_rd_final<R>), dim3((sh.by + RdLine<R>::N - 1) / RdLine<R>::N, n), dim3(RdLine<R>::NT), 0, s, a)
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
