"""The bounce solvers on the aperture's window (circular convolutions of 16 R points per
line) against the transforms of the whole grid: every radix, windows at the edge of a
radix and of the grid, rectangular grids, tilts and surfaces, given emission and
reflection, batches of frequencies, replayed graphs, k ranges without a mirror
symmetry; and against the CPU oracle."""
import numpy as np
import pytest

import BoostFractor as B
from BoostFractor import workloads as W
from helpers import DISKR, O, ocoords, osetup, rel

pytestmark = pytest.mark.gpu
# whole-grid and windowed transforms round differently by ~1e-15 per bounce; fields stored
# in complex64 round at 6e-8 of their maximum per pass
TOL = {"fp64": 1e-12, "mixed": 2e-6}


def _both(fn):
    out = []
    for on in (2, 0):  # 2: on the window however few the bounces
        with B.context().options(reduced=on):
            out.append(fn())
    return out


def _grid(nx, ny, shift=0):
    def axis(n):
        return (np.arange(n) - n // 2 + shift) / 128.0
    X, Y = axis(nx), axis(ny)
    k = lambda v: (np.arange(len(v)) - (len(v) - 1) / 2.0) * 2 * np.pi / (len(v) / 128.0)  # noqa: E731
    return B.CoordinateSystem(X, Y, k(X), k(Y))


def _booster(c, rough, seed):
    sb = W.rough_booster(c, ndisk=2, seed=seed) if rough else W.booster(c, ndisk=2, seed=seed)
    return sb


# radius in samples of 1/128 m: bands of 2 r - 1 .. 2 r + 1 samples, radices 4, 5, 6, 8, 10, 12, 16, 20
@pytest.mark.parametrize("radius", [3.2, 16.0, 16.6, 20.4, 24.0, 24.3, 32.4, 40.3, 48.5, 63.9, 64.2, 79.9])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_dancer_on_every_radix(radius, prec):
    n = 128 if radius < 32 else 256 if radius < 64 else 512
    c = _grid(n, n)
    sb = _booster(c, False, 11)
    R = radius / 128.0
    a, b = _both(lambda: B.dancer(0, 9, sb, c, f=[19.8e9, 20.2e9], diskR=R, precision=prec))
    assert np.any(b != 0) and rel(a, b) < TOL[prec]


@pytest.mark.parametrize("nx,ny,shift", [(128, 256, 0), (101, 130, 0), (150, 100, 0), (256, 128, 30), (200, 120, -58),
                                         (97, 512, 5)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_dancer_on_other_grids_and_windows(nx, ny, shift, prec):
    """rectangular grids; windows off the centre, cut by the grid's edge"""
    c = _grid(nx, ny, shift)
    sb = _booster(c, True, 12)
    refl = np.exp(-(c.X[None] ** 2 + c.Y[:, None] ** 2) / 0.1 ** 2) * np.exp(3j * c.X[None])
    rng = np.random.default_rng(3)
    emit = rng.standard_normal((len(sb.distance) - 1, 2, ny, nx)) + 0j
    for kw in ({}, {"reflect": refl}, {"emit": emit}):
        a, b = _both(lambda: B.dancer(0, 8, sb, c, f=[20e9], diskR=DISKR, precision=prec, **kw))
        assert np.any(b != 0) and rel(a, b) < TOL[prec]
    a, b = _both(lambda: B.dancer(0, 8, sb, c, f=20e9, prop=B.propagatorNoTilts, diskR=DISKR, precision=prec))
    assert rel(a, b) < TOL[prec]


def _shifted(c, kx, ky):
    """k axes moved by fractions of a step: their phases are no longer even, the tables no quarters"""
    k = lambda v, d: v + d * (v[1] - v[0])  # noqa: E731
    return B.CoordinateSystem(c.X, c.Y, k(c.kX, kx), k(c.kY, ky))


@pytest.mark.parametrize("nx,ny", [(128, 128), (101, 101), (128, 101)])
@pytest.mark.parametrize("kx,ky", [(0.3, 0.0), (0.0, -0.4), (0.5, 0.2)])
def test_k_ranges_without_mirror_symmetry(nx, ny, kx, ky):
    c = _shifted(_grid(nx, ny), kx, ky)
    sb = _booster(c, True, 16)
    f = [19.9e9, 20.2e9]
    a, b = _both(lambda: B.dancer(0, 9, sb, c, f=f, diskR=DISKR))
    assert np.any(b != 0) and rel(a, b) < TOL["fp64"]
    for q in range(len(f)):
        assert rel(a[q], O.dancer(osetup(sb), ocoords(c), 0, 9, f[q], diskR=DISKR)) < 1e-10
    sb.r[0] = 0.7 + 0.1j
    for prec in ("fp64", "mixed"):
        x, y = _both(lambda: B.cheerleader(0, 8, sb, c, f=f, diskR=DISKR, precision=prec, returnboth=True))
        for u, v in zip(x, y):
            assert np.any(v != 0) and rel(u, v) < TOL[prec]
        if prec == "fp64":
            for q in range(len(f)):
                want = O.cheerleader(osetup(sb), ocoords(c), 0, 8, f[q], diskR=DISKR, returnboth=True)
                assert all(rel(u[q], v) < 1e-10 for u, v in zip(x, want))


@pytest.mark.parametrize("nx,ny,shift", [(128, 128, 0), (101, 130, 0), (256, 128, 30)])
def test_window_matches_oracle(nx, ny, shift):
    """symmetric k ranges (quarter tables), even and odd, a window off the centre: emission, reflection"""
    c = _grid(nx, ny, shift)
    sb = _booster(c, True, 17)
    os_, oc = osetup(sb), ocoords(c)
    refl = np.exp(-(c.X[None] ** 2 + c.Y[:, None] ** 2) / 0.1 ** 2) * np.exp(3j * c.X[None])
    for kw in ({}, {"reflect": refl}):
        with B.context().options(reduced=2):
            got = B.dancer(0, 9, sb, c, f=20.1e9, diskR=DISKR, **kw)
        assert rel(got, O.dancer(os_, oc, 0, 9, 20.1e9, diskR=DISKR, **kw)) < 1e-10
        got = B.cheerleader(0, 8, sb, c, f=20.1e9, diskR=DISKR, **kw)
        assert rel(got, O.cheerleader(os_, oc, 0, 8, 20.1e9, diskR=DISKR, **kw)) < 1e-10


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_dancer_plans_batches_and_graphs(prec):
    c = _grid(128, 128)
    sb = _booster(c, True, 13)
    f = np.linspace(19.5e9, 20.5e9, 7)
    want = B.dancer(0, 10, sb, c, f=f, diskR=DISKR, precision=prec)  # 11 bounces: on the window
    for graph in (0, 1):
        with B.context().options(graph=graph):
            plan = B.DancerPlan(0, 10, sb, c, f, diskR=DISKR, precision=prec, freq_batch=3)
            for _ in range(3):
                plan.run()
                B.dancer(0, 8, sb, c, f=20e9, diskR=DISKR)  # eager work on the same stream in between
                E, power = plan.fetch()
                assert np.array_equal(E, want)
                assert np.allclose(power, np.sum(np.abs(want) ** 2, axis=(1, 2)), rtol=1e-12)
            plan.close()


def test_plan_timing_counts_the_launches():
    c = _grid(128, 128)
    sb = _booster(c, False, 20)
    for reduced, rows in ((0, 12), (1, 11)):  # the window's last bounce ends with the sum of the exit fields
        with B.context().options(reduced=reduced):
            plan = B.DancerPlan(0, 11, sb, c, np.linspace(19.8e9, 20.2e9, 6), diskR=DISKR, freq_batch=3)
            plan.timing(True)
            plan.run()
            kt = plan.kernel_times()
            plan.close()
        assert kt["col_pass"][1] == 2 * 12 and kt["row_pass"][1] == 2 * rows
        assert kt["col_pass"][0] > 0 and kt["row_pass"][0] > 0


@pytest.mark.parametrize("tilted", [False, True])
def test_dancer_batch_is_bounded_by_its_whole_grid_tables(tilted):
    """a small window on a fine grid: the batch's phase and tilt tables are on the whole grid"""
    n, R = 1024, 0.02
    c = W.grid_coords(n)
    sb = W.booster(c, ndisk=20, seed=15, flat=True)
    nreg = len(sb.distance)
    if tilted:
        sb.relative_tilt_x = np.full(nreg, 1e-4)
    f = np.linspace(19e9, 21e9, 64)
    with B.context().options(reduced=1):
        plan = B.DancerPlan(0, 9, sb, c, f, diskR=R)
        fb = plan.freq_batch
        plan.close()
    tables = 16 * n * n * (20 + (nreg - 1 if tilted else 0))  # at least: 20 gaps of their own, tilts
    assert 1 <= fb and fb * tables <= 2 << 30


def _by_rule(fn):
    """the default's choice of the path, and the whole grid"""
    out = []
    for on in (1, 0):
        with B.context().options(reduced=on):
            out.append(fn())
    return out


@pytest.mark.parametrize("n,ndisk,nfreq,window_from", [(128, 1, 1, 11), (101, 3, 1, 11), (256, 2, 1, 11),
                                                       (128, 9, 2, 8), (101, 9, 1, 8), (256, 9, 1, 8)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_few_fields_take_the_window_later(n, ndisk, nfreq, window_from, prec):
    """8 to 10 bounces of few fields are faster on the whole grid; with the same FP64 fields"""
    c = W.grid_coords(n)
    sb = W.booster(c, ndisk=ndisk, seed=18)
    f = np.linspace(19.9e9, 20.1e9, nfreq)
    for nmax in (6, 7, 9, 10, 14):
        with B.context().options(reduced=0):
            grid = B.dancer(0, nmax, sb, c, f=f, diskR=DISKR, precision="mixed" if nmax == 6 else "fp64")
        got = B.dancer(0, nmax, sb, c, f=f, diskR=DISKR, precision="mixed" if nmax == 6 else prec)
        assert rel(got, grid) < TOL["fp64"]
        assert np.array_equal(got, grid) == (nmax + 1 < window_from)


def test_short_runs_on_the_window():
    """option reduced=2: one, two and four bounces"""
    c = _grid(128, 101)
    sb = _booster(c, True, 19)
    for nmax in (0, 1, 3):
        for fn in (lambda: B.dancer(0, nmax, sb, c, f=[19.9e9, 20.1e9], diskR=DISKR),
                   lambda: B.cheerleader(0, nmax, sb, c, f=[19.9e9, 20.1e9], diskR=DISKR)):
            a, b = _both(fn)
            assert np.any(b != 0) and rel(a, b) < TOL["fp64"]


def test_history_amin_and_short_runs_keep_the_whole_grid():
    c = _grid(128, 128)
    sb = _booster(c, False, 14)
    for kw in ({"returnsum": False, "immediatesum": False}, {"returnsum": True, "immediatesum": False}):
        a, b = _by_rule(lambda: B.dancer(0, 9, sb, c, f=20e9, diskR=DISKR, **kw))
        assert np.array_equal(a, b)
    a, b = _by_rule(lambda: B.dancer(0.05, 30, sb, c, f=20e9, diskR=DISKR))
    assert np.array_equal(a, b)
    a, b = _by_rule(lambda: B.dancer(0, 3, sb, c, f=20e9, diskR=DISKR))
    assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,ny,shift", [(128, 128, 0), (101, 101, 0), (256, 128, 30), (150, 100, 0)])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("ndisk", [1, 3])
def test_cheerleader_on_the_window(nx, ny, shift, prec, ndisk):
    c = _grid(nx, ny, shift)
    sb = W.rough_booster(c, ndisk=ndisk, seed=21)
    refl = np.exp(-(c.X[None] ** 2 + c.Y[:, None] ** 2) / 0.1 ** 2) * np.exp(3j * c.X[None])
    rng = np.random.default_rng(4)
    emit = rng.standard_normal((len(sb.distance), 2, ny, nx)) + 1j * rng.standard_normal((len(sb.distance), 2, ny, nx))
    sb.r[0] = 0.7 + 0.1j  # so that something leaves on the left
    for kw in ({}, {"reflect": refl}, {"emit": emit}):
        a, b = _both(lambda: B.cheerleader(0, 9, sb, c, f=[19.9e9, 20e9, 20.3e9], diskR=DISKR, precision=prec,
                                           returnboth=True, **kw))
        for x, y in zip(a, b):
            assert np.any(y != 0) and rel(x, y) < TOL[prec]
    a, b = _both(lambda: B.cheerleader(0, 9, sb, c, f=20e9, prop=B.propagatorNoTilts, diskR=DISKR, precision=prec))
    assert rel(a, b) < TOL[prec]


def test_cheerleader_amin_and_short_runs_keep_the_whole_grid():
    c = _grid(128, 128)
    sb = _booster(c, False, 22)
    a, b = _by_rule(lambda: B.cheerleader(0.05, 30, sb, c, f=20e9, diskR=DISKR))
    assert np.array_equal(a, b)
    a, b = _by_rule(lambda: B.cheerleader(0, 2, sb, c, f=20e9, diskR=DISKR))
    assert np.array_equal(a, b)
