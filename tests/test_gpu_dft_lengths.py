"""Line transforms of lengths that are no power of two, on the matrix cores:
edges of the 16-wide output tiles, of the quarters of the contraction, of the
waves of a block and of its LDS, against numpy's transforms and against the
direct transforms in LDS (option fft_lds)."""
import numpy as np
import pytest

import BoostFractor as B
from BoostFractor import workloads as W
from helpers import DISKR, rel

pytestmark = pytest.mark.gpu

# a transform of n points sums n/2 products per output: rounding of a propagation
# (four transforms) stays below 4 (n/2 + 8) eps of the field's 1-norm per line; with
# random fields that is within a small multiple of sqrt(n) eps of the maximum
EPS = 2.0 ** -52


def _axis(n):
    return (np.arange(n) - n // 2) / max(n, 2)


def _coords(nx, ny):
    def k(X):
        return (np.arange(len(X)) - (len(X) - 1) / 2.0) * 6.0
    X, Y = _axis(nx), _axis(ny)
    return B.CoordinateSystem(X, Y, k(X), k(Y))


def _propagate(E, c, dz, R, k0, tilt, surface):
    """mask, FFT, exp(-i kz dz), inverse FFT, tilt, surface (real permittivity)"""
    mask = np.abs(c.X[None] ** 2 + c.Y[:, None] ** 2) < R * R
    kx, ky = np.roll(c.kX, -(c.nx // 2)), np.roll(c.kY, -(c.ny // 2))
    arg = k0 * k0 - kx[None] ** 2 - ky[:, None] ** 2
    kz = np.sqrt(np.abs(arg))
    ph = np.where(arg >= 0, np.exp(-1j * kz * dz), np.exp(-kz * dz))
    T = np.fft.ifft2(np.fft.fft2(E * mask) * ph)
    return T * np.exp(-1j * k0 * (tilt[0] * c.X[None] + tilt[1] * c.Y[:, None] + surface))


@pytest.mark.parametrize("nx,ny", [(1, 3), (2, 15), (7, 17), (31, 31), (33, 30), (47, 63), (65, 34), (96, 97),
                                   (127, 129), (101, 128), (64, 255), (257, 9), (9, 511), (513, 12), (12, 1023),
                                   (1000, 7)])
@pytest.mark.parametrize("R", [0.15, 5.0])
def test_propagation_of_any_length(nx, ny, R):
    rng = np.random.default_rng(nx * 1031 + ny)
    c = _coords(nx, ny)
    E = rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))
    S = 1e-4 * rng.standard_normal((ny, nx))
    k0 = 2 * np.pi / 0.015
    want = _propagate(E, c, 3e-3, R, k0, (1e-3, -2e-3), S)
    got = B.propagator(E, 3e-3, R, 1.0, 1e-3, -2e-3, S, 0.015, c)
    # the phases k0 S and kz dz (up to ~10) carry ~10 eps of their own
    assert np.max(np.abs(got - want)) <= (40 + 16 * np.sqrt(max(nx, ny))) * EPS * np.max(np.abs(E)) * 4


@pytest.mark.parametrize("n,prec", [(101, "fp64"), (101, "mixed"), (30, "fp64"), (52, "mixed"), (129, "fp64")])
@pytest.mark.parametrize("rough", [False, True])
@pytest.mark.parametrize("reduced", [0, 2], ids=["grid", "window"])
def test_dancer_any_length_matches_direct_transforms(n, prec, rough, reduced):
    """summed, history and amin runs against the direct transforms; skipping the
    rows that the aperture zeroes changes no bit (on the whole grid; the summed run's window, where the grid
    has one, against the same direct transforms)"""
    coords = W.grid_coords(n)
    sb = W.rough_booster(coords, ndisk=2, seed=77) if rough else W.booster(coords, ndisk=3, seed=78)
    freqs = [19.8e9, 20.1e9, 20.3e9]
    out = {}
    for key, o in (("mm", {}), ("lds", {"fft_lds": 1}), ("rows", {"band": 0})):
        with B.context().options(reduced=reduced, **o):
            out[key] = [B.dancer(0, 12, sb, coords, f=freqs, diskR=DISKR, precision=prec),
                        B.dancer(0, 5, sb, coords, f=20e9, diskR=DISKR, precision=prec, returnsum=False,
                                 immediatesum=False),
                        B.dancer(0.05, 30, sb, coords, f=20e9, diskR=DISKR, precision=prec)]
    # fields stored in complex64 round differently in every bounce
    tol = {"fp64": 1e-12, "mixed": 1e-5}[prec]
    for q in range(3):
        assert np.any(out["mm"][q] != 0)
        assert rel(out["mm"][q], out["lds"][q]) < tol
        assert np.array_equal(out["mm"][q], out["rows"][q])


@pytest.mark.parametrize("n,prec", [(101, "fp64"), (101, "mixed"), (37, "fp64"), (130, "fp64")])
@pytest.mark.parametrize("opt", [{}, {"chwave": 0}, {"chxf": 0}, {"chfuse": 0}, {"band": 0}])
def test_cheerleader_any_length_matches_direct_transforms(n, prec, opt):
    coords = W.grid_coords(n)
    sb = W.rough_booster(coords, ndisk=2, seed=79)
    freqs = [19.8e9, 20.1e9]
    refl = np.exp(-(coords.X[None] ** 2 + coords.Y[:, None] ** 2) / 0.1 ** 2).astype(complex)
    with B.context().options(fft_lds=1):
        want = [B.cheerleader(0, 6, sb, coords, f=freqs, diskR=DISKR, precision=prec),
                B.cheerleader(0.05, 20, sb, coords, f=20e9, reflect=refl, diskR=DISKR, precision=prec)]
    with B.context().options(**opt):
        got = [B.cheerleader(0, 6, sb, coords, f=freqs, diskR=DISKR, precision=prec),
               B.cheerleader(0.05, 20, sb, coords, f=20e9, reflect=refl, diskR=DISKR, precision=prec)]
    tol = {"fp64": 1e-12, "mixed": 1e-5}[prec]
    for g, w in zip(got, want):
        assert np.any(w != 0) and rel(g, w) < tol


@pytest.mark.parametrize("n,direct", [(7, True), (24, True), (31, True), (33, False)])
def test_short_lines_with_the_amin_criterion(n, direct):
    """one region at a time on lines below 32 points: the direct sums in LDS, bit for bit"""
    coords = W.grid_coords(n)
    sb = W.rough_booster(coords, ndisk=2, seed=81)
    out = []
    for lds in (0, 1):
        with B.context().options(fft_lds=lds):
            out.append(B.cheerleader(1e-6, 12, sb, coords, f=[19.8e9, 20.1e9], diskR=0.3))
    assert np.any(out[1] != 0) and rel(out[0], out[1]) < 1e-12
    assert np.array_equal(out[0], out[1]) == direct


def test_empty_aperture_gives_a_zero_field():
    c = _coords(30, 21)
    c.X[:] += 0.5 / 30  # no sample at the centre
    E = np.ones((21, 30), dtype=complex)
    assert not np.any(B.propagator(E, 3e-3, 1e-6, 1.0, 0, 0, None, 0.015, c))


def test_more_lengths_than_the_context_keeps_tables_of():
    """the context keeps the matrices of the last lengths; a plan holds its own"""
    coords = W.grid_coords(50)
    sb = W.booster(coords, ndisk=2, seed=80)
    plan = B.DancerPlan(0, 8, sb, coords, [20e9], diskR=DISKR)
    plan.run()
    first = plan.fetch()[0]
    for n in range(20, 31):
        c = _coords(n, n)
        B.propagator(np.ones((n, n), dtype=complex), 1e-3, DISKR, 1.0, 0, 0, None, 0.015, c)
    plan.run()
    assert np.array_equal(plan.fetch()[0], first)
    plan.close()
