"""Parseval products over a band of frequencies, interpolated in k0^2 at
Chebyshev nodes (option parseval_nodes), against the direct products and the
CPU oracle.  Narrow and wide bands, gaps of 0 to 0.4 m (waves that propagate
grow on the interpolation's ellipse with the gap), grids with few and many
k-bin groups, frequencies in any order and repeated, and gaps the
interpolation has to leave alone: a lossy one and, with the propagator that
keeps it, a permittivity with imaginary part +0.
"""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import BoostFractor as B
from BoostFractor import workloads as W
from helpers import DISKR, O, ocoords, rel
from test_gpu_support import _modes

pytestmark = pytest.mark.gpu


def _stack(n, eps):
    """gaps of several lengths, one of them with its own permittivity"""
    coords = W.grid_coords(n)
    dist = np.array([0.0, 8e-3, 1e-3, 0.0, 1e-3, 2.5e-2, 1e-3, 0.4, 1e-3, 7.9e-3])
    e = np.array([np.nan, 1, 24, 1, 24, 1, 24, 1, 24, eps], dtype=complex)
    return coords, B.SeedSetupBoundaries(coords, diskno=4, distance=dist, epsilon=e)


@pytest.mark.parametrize("lo,hi,nf", [(19.99e9, 20.01e9, 40), (19.5e9, 20.5e9, 100), (12e9, 24e9, 64), (20e9, 20.2e9, 9)])
@pytest.mark.parametrize("n", [33, 128])
@pytest.mark.parametrize("kind", [(B.propagator, O.PROP_PROPAGATOR), (B.propagatorNoTilts, O.PROP_NOTILTS)],
                         ids=["propagator", "notilts"])
def test_interpolated_products(engine_options, n, lo, hi, nf, kind):
    coords, sb = _stack(n, complex(1.0, -1e-3))
    modes = _modes(coords, DISKR)
    freqs = np.random.default_rng(nf).permutation(np.append(np.linspace(lo, hi, nf - 1), lo))
    gaps = [1, 3, 5, 7, 9]
    got = B.calc_propagation_matrices(sb, coords, modes, f=freqs, prop=kind[0], diskR=DISKR)
    engine_options(parseval_nodes=0)
    want = B.calc_propagation_matrices(sb, coords, modes, f=freqs, prop=kind[0], diskR=DISKR)
    for q in range(nf):
        for r in gaps:
            assert rel(got[q][r], want[q][r]) < 1e-13, (q, r, rel(got[q][r], want[q][r]))
    pat, kt = modes.patterns_flat()[:, 0], modes.mode_kt.reshape(-1)
    for q in (0, nf // 2):
        for r in gaps:
            o = O.propagation_matrix(sb.distance[r], DISKR, sb.eps[r], 0.0, 0.0, np.zeros((n, n), dtype=complex),
                                     B.wavelength(freqs[q]), ocoords(coords), pat, kt, kind[1])
            assert rel(got[q][r], o) < 1e-10, (q, r)


def test_weight_tables_are_bounded():
    """a fine grid with many gaps: the interpolation's weight tables (131 000 groups x 40 gaps x 10 to 20
    nodes, 0.8 GB in one) are formed in parts of 512 MB, and the parts add up"""
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded
    coords = W.grid_coords(1024)
    sb = W.booster(coords, ndisk=40, spacings=np.linspace(5e-3, 12e-3, 40), flat=True)
    modes = _modes(coords, DISKR)
    freqs = np.linspace(19.5e9, 20.5e9, 64)

    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    def run(nodes):
        ctx = B.context()  # of a thread of its own
        ctx.set_option("parseval_nodes", nodes)
        before = free_bytes()
        P = B.calc_propagation_matrices(sb, coords, modes, f=freqs, diskR=DISKR)
        kept = before - free_bytes()
        ctx.close()
        return np.asarray([[P[q][r] for r in range(1, 81, 2)] for q in range(len(freqs))]), kept

    def fresh(nodes):
        with ThreadPoolExecutor(max_workers=1) as ex:
            return ex.submit(run, nodes).result()

    fresh(0)  # code objects and the runtime's own buffers
    want, base = fresh(0)
    got, kept = fresh(1)
    assert np.any(got != want)  # (interpolated)
    for q in range(len(freqs)):
        for r in range(40):
            assert rel(got[q][r], want[q][r]) < 1e-13, (q, r, rel(got[q][r], want[q][r]))
    assert kept - base <= (512 << 20) + (128 << 20)
