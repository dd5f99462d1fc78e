"""Disk matrices summed over the points where the patterns are not zero.

Patterns that vanish outside the aperture (the Bessel modes) take the sums over
their support, patterns on the whole grid the sums over the grid, patterns that
reach a little beyond the aperture the support with separately masked
transforms.  Each against the CPU oracle at the suite's 1e-10, with one or two
frequencies (a weight table per frequency) and a band (moments of the heights).
"""
import numpy as np
import pytest

import BoostFractor as B
from BoostFractor import workloads as W
from helpers import DISKR, O, ocoords, rel

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _modes(coords, radius):
    """three complex patterns inside `radius`"""
    XX, YY = np.meshgrid(coords.X, coords.Y)
    r, phi = np.hypot(XX, YY), np.arctan2(YY, XX)
    pat = np.zeros((1, 3, 1, coords.ny, coords.nx), dtype=complex)
    for q, l in enumerate((-1, 0, 1)):
        p = np.exp(-(r / 0.1) ** 2 - 1j * l * phi) * (r / 0.1) ** abs(l) * (r <= radius)
        pat[0, q, 0] = p / np.linalg.norm(p)
    kt = np.array([[25.5 + 0j, 16.0 + 0j, 25.5 + 0j]])
    return B.SeedModes(coords, ThreeDim=True, Mmax=1, Lmax=1, pattern_input=pat, kT_arr=kt)


def _booster(n, seed):
    coords = W.grid_coords(n)
    sb = W.booster(coords, ndisk=2, seed=seed)
    nreg = len(sb.distance)
    rng = np.random.default_rng(seed)
    sb.relative_tilt_x, sb.relative_tilt_y = 1e-4 * rng.standard_normal(nreg), 1e-4 * rng.standard_normal(nreg)
    surf = np.zeros((nreg, n, n), dtype=complex)
    surf[2] = 1e-5 * rng.standard_normal((n, n))
    surf[4] = 1e-5 * rng.standard_normal((n, n))
    sb.relative_tilt_x[4] = sb.relative_tilt_y[4] = 0.0
    sb.relative_surfaces = surf
    return coords, sb


def _check(sb, coords, modes, freqs, regions):
    got = B.calc_propagation_matrices(sb, coords, modes, f=freqs, diskR=DISKR)
    pat, kt = modes.patterns_flat()[:, 0], modes.mode_kt.reshape(-1)
    for q in {0, len(freqs) - 1}:
        for r in regions:
            want = O.propagation_matrix(sb.distance[r], DISKR, sb.eps[r], sb.relative_tilt_x[r], sb.relative_tilt_y[r],
                                        sb.relative_surfaces[r], B.wavelength(freqs[q]), ocoords(coords), pat, kt,
                                        O.PROP_PROPAGATOR)
            assert rel(got[q][r], want) < TOL, (q, r, rel(got[q][r], want))
    return got


@pytest.mark.parametrize("radius", [DISKR, 0.2, 2.0])
@pytest.mark.parametrize("nf", [1, 2, 12])
@pytest.mark.parametrize("n", [48, 65])
def test_disk_matrices_on_the_support(n, nf, radius):
    coords, sb = _booster(n, 40 + n)
    _check(sb, coords, _modes(coords, radius), np.linspace(19.8e9, 20.2e9, nf), (2, 4))


@pytest.mark.parametrize("nf", [1, 12])
def test_heights_off_the_support(nf):
    """large heights where no pattern reaches change nothing; a lossy disk whose weights overflow there and
    heights that are not finite give NaN as the sums over the grid do"""
    coords, sb = _booster(48, 5)
    modes = _modes(coords, DISKR)
    freqs = np.linspace(19.8e9, 20.2e9, nf)
    sb.relative_surfaces[4, 0, 0] = 3e-3
    base = _check(sb, coords, modes, freqs, (2, 4))
    lossy = sb.copy()
    lossy.eps[4] = 24.0 - 0.5j
    lossy.relative_surfaces[4, 0, 0] = -1e3
    bad = sb.copy()
    bad.relative_surfaces[4, 0, 0] = np.nan
    for s in (lossy, bad):
        got = B.calc_propagation_matrices(s, coords, modes, f=freqs, diskR=DISKR)
        assert not np.isfinite(got[0][4]).any() and rel(got[0][2], base[0][2]) < 1e-12
