"""The register DFTs of the reduced propagation (boostfractor.jl_amd/csrc/bf_fftmix.h)
on the CPU: every radix, forward and inverse, half of the inputs zero or half of the
outputs formed, against the direct sum; and the two-pass lines of 16 R points built
from them (radix R, twiddles, radix 16, and back) against numpy's transforms."""
import os
import shutil
import subprocess

import pytest

from test_fft_pruning_cpu import _host_copy

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "boostfractor.jl_amd", "csrc")

MAIN = r'''
#include <cmath>
#include <complex>
#include <cstdio>
#include <type_traits>
template <typename T> struct alignas(2 * sizeof(T)) cplx { T re, im; };
typedef cplx<double> zd;
template <typename T> inline cplx<T> cmk(T a, T b) { cplx<T> z; z.re = a; z.im = b; return z; }
template <typename T> inline cplx<T> cadd(cplx<T> a, cplx<T> b) { return cmk<T>(a.re + b.re, a.im + b.im); }
template <typename T> inline cplx<T> csub(cplx<T> a, cplx<T> b) { return cmk<T>(a.re - b.re, a.im - b.im); }
template <typename T> inline cplx<T> cmul(cplx<T> a, cplx<T> b) { return cmk<T>(a.re*b.re - a.im*b.im, a.re*b.im + a.im*b.re); }
template <typename To, typename Ti> inline cplx<To> ccast(cplx<Ti> a) { return cmk<To>((To)a.re, (To)a.im); }
template <typename T, bool INV> inline cplx<T> tw_get(const cplx<T>* tw, int m) { return tw[m]; }
template <typename T, bool INV> inline void radix4(cplx<T>& a0, cplx<T>& a1, cplx<T>& a2, cplx<T>& a3) {
    cplx<T> t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = csub(a1, a3);
    t3 = INV ? cmk<T>(-t3.im, t3.re) : cmk<T>(t3.im, -t3.re);
    a0 = cadd(t0, t2); a2 = csub(t0, t2); a1 = cadd(t1, t3); a3 = csub(t1, t3);
}
inline void __syncthreads() {}
using std::fma;
#include FFTREG_HOST
#include FFTMIX_HOST
typedef std::complex<double> C;
static unsigned long long st = 12345;
static double rnd() { st = st * 6364136223846793005ull + 1442695040888963407ull; return (double)(st >> 11) / 9007199254740992.0 - 0.5; }
static double worst = 0;
static C w(int k, int n) { const double t = 2 * M_PI * (double)(((k % n) + n) % n) / n; return C(std::cos(t), std::sin(t)); }
template <int R, bool INV> void one() {
    constexpr int H = bf::rd_half(R);
    zd a[R], b[R];
    for (int m = 0; m < R; m++) { a[m] = m < H ? cmk<double>(rnd(), rnd()) : cmk<double>(NAN, NAN); b[m] = cmk<double>(rnd(), rnd()); }
    zd x[R], y[R];
    for (int m = 0; m < R; m++) { x[m] = a[m]; y[m] = b[m]; }
    bf::dft_in<R, INV>(x);
    bf::dft_out_half<R, INV>(y);
    for (int k = 0; k < R; k++) {
        C s = 0, t = 0;
        for (int m = 0; m < R; m++) {
            if (m < H) s += C(a[m].re, a[m].im) * w(INV ? m * k : -m * k, R);
            t += C(b[m].re, b[m].im) * w(INV ? m * k : -m * k, R);
        }
        worst = std::fmax(worst, std::abs(s - C(x[k].re, x[k].im)));
        if (k < H) worst = std::fmax(worst, std::abs(t - C(y[k].re, y[k].im)));
    }
}
// a line of M = 16 R points: thread t of 16 holds t + 16 m, thread k1 of R holds k1 + R k2
template <int R> void line() {
    constexpr int M = 16 * R, H = bf::rd_half(R);
    const int band = (M + 1) / 2;
    C x[M], X[M], z[16][R];
    for (int i = 0; i < M; i++) x[i] = i < band ? C(rnd(), rnd()) : C(0, 0);
    for (int t = 0; t < 16; t++) {
        zd a[R];
        for (int m = 0; m < R; m++) a[m] = m < H ? cmk<double>(x[t + 16 * m].real(), x[t + 16 * m].imag()) : cmk<double>(0, 0);
        bf::dft_in<R, false>(a);
        for (int k1 = 0; k1 < R; k1++) z[t][k1] = C(a[k1].re, a[k1].im) * w(-t * k1, M);
    }
    for (int k1 = 0; k1 < R; k1++) {
        zd v[16];
        for (int t = 0; t < 16; t++) v[t] = cmk<double>(z[t][k1].real(), z[t][k1].imag());
        bf::dft_reg<double, 16, false>(v);
        for (int k2 = 0; k2 < 16; k2++) X[k1 + R * k2] = C(v[k2].re, v[k2].im);
        bf::dft_reg<double, 16, true>(v);
        for (int t = 0; t < 16; t++) z[t][k1] = C(v[t].re, v[t].im);
    }
    for (int k = 0; k < M; k++) {
        C s = 0;
        for (int i = 0; i < M; i++) s += x[i] * w(-i * k, M);
        worst = std::fmax(worst, std::abs(s - X[k]) / 16);
    }
    for (int t = 0; t < 16; t++) {
        zd a[R];
        for (int k1 = 0; k1 < R; k1++) { const C v = z[t][k1] * w(t * k1, M); a[k1] = cmk<double>(v.real(), v.imag()); }
        bf::dft_out_half<R, true>(a);
        for (int m = 0; m < H; m++)
            if (t + 16 * m < band) worst = std::fmax(worst, std::abs(C(a[m].re, a[m].im) / (double)M - x[t + 16 * m]));
    }
}
template <int R> void all() { one<R, false>(); one<R, true>(); line<R>(); std::printf("%d %g\n", R, worst); }
int main() { all<4>(); all<5>(); all<6>(); all<8>(); all<10>(); all<12>(); all<16>(); all<20>(); std::printf("worst %g\n", worst); return worst < 2e-14 ? 0 : 1; }
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_half_transforms_match_direct_sums(tmp_path):
    for h in ("bf_fftreg.h", "bf_fftmix.h"):
        text = _host_copy(open(os.path.join(CSRC, h)).read()).replace('#include "bf_fftreg.h"', "")
        (tmp_path / h).write_text(text)
    src = tmp_path / "main.cpp"
    src.write_text(MAIN)
    exe = tmp_path / "main"
    subprocess.run(["g++", "-O1", "-std=c++17", f'-DFFTREG_HOST="{tmp_path / "bf_fftreg.h"}"',
                    f'-DFFTMIX_HOST="{tmp_path / "bf_fftmix.h"}"', str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
