"""Device memory that a context keeps for its next calls: results do not depend on
what an earlier call left in it, threads with contexts of their own do not meet,
and destroying the context gives the memory back."""
import ctypes
import threading

import numpy as np
import pytest

import BoostFractor as B
from BoostFractor import workloads as W
from helpers import DISKR

pytestmark = pytest.mark.gpu


def _calls(n):
    coords = W.grid_coords(n)
    sb = W.booster(coords, ndisk=2, seed=90)
    modes = B.SeedModes(coords, ThreeDim=True, Mmax=2, Lmax=1, diskR=DISKR)
    E = np.exp(-(coords.X[None] ** 2 + coords.Y[:, None] ** 2) / 0.1 ** 2).astype(complex)
    return [B.propagator(E, 4e-3, DISKR, 9.0, 1e-4, 0.0, None, 0.015, coords),
            B.dancer(0, 6, sb, coords, f=[19.9e9, 20.1e9], diskR=DISKR),
            B.cheerleader(0, 5, sb, coords, f=20e9, diskR=DISKR),
            B.transformer(sb.copy(), coords, modes, f=[19.9e9, 20.1e9], diskR=DISKR)]


def test_results_do_not_depend_on_earlier_calls():
    sizes = [64, 30, 48, 64]
    first = {}
    for _ in range(2):
        for n in sizes:
            got = _calls(n)
            for g, w in zip(got, first.setdefault(n, got)):
                assert np.array_equal(g, w)


def test_threads_with_their_own_contexts():
    want = {n: _calls(n) for n in (32, 40, 64)}
    bad = []

    def work(n):
        try:
            for _ in range(5):
                for g, w in zip(_calls(n), want[n]):
                    if not np.array_equal(g, w):
                        bad.append(n)
        except Exception as e:  # noqa: BLE001 (reported below)
            bad.append(e)

    ts = [threading.Thread(target=work, args=(n,)) for n in want]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_a_plan_outlives_other_plans_of_its_context():
    coords = W.grid_coords(64)
    sb = W.booster(coords, ndisk=2, seed=91)
    plan = B.DancerPlan(0, 10, sb, coords, [19.9e9, 20.1e9], diskR=DISKR)
    plan.run()
    want = plan.fetch()[0]
    for _ in range(4):
        other = B.DancerPlan(0, 3, sb, coords, [20e9, 20.2e9], diskR=DISKR)
        other.run()
        other.close()
        plan.run()
        assert np.array_equal(plan.fetch()[0], want)
    plan.close()


def test_destroying_a_context_gives_its_memory_back():
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded

    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    coords = W.grid_coords(256)
    sb = W.booster(coords, ndisk=8, seed=92, flat=True)

    def used_by_a_context():
        ctx = B.Context()
        before = free_bytes()
        plan = B.DancerPlan(0, 1, sb, coords, np.linspace(19e9, 21e9, 16), diskR=DISKR, ctx=ctx)
        plan.run()
        ctx.synchronize()
        plan.close()
        kept = before - free_bytes()
        ctx.close()
        return before, kept

    used_by_a_context()  # code objects and the runtime's own buffers
    before, kept = used_by_a_context()
    assert free_bytes() >= before - (8 << 20)
    assert kept <= (2 << 30) + (64 << 20)


def test_memory_given_back_on_request():
    """option pool_mb: 0 frees what the context keeps and keeps nothing more; the results are the same"""
    hip = ctypes.CDLL("libamdhip64.so")  # the runtime the library has loaded

    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    coords = W.grid_coords(256)
    sb = W.booster(coords, ndisk=8, seed=93, flat=True)
    ctx = B.Context()

    def run():
        plan = B.DancerPlan(0, 1, sb, coords, np.linspace(19e9, 21e9, 16), diskR=DISKR, ctx=ctx)
        plan.run()
        E = plan.fetch()[0]
        plan.close()
        return E

    want = run()
    ctx.set_option("pool_mb", 0)
    empty = free_bytes()
    assert np.array_equal(run(), want)
    assert free_bytes() >= empty - (8 << 20)
    ctx.set_option("pool_mb", 2048)
    assert np.array_equal(run(), want)
    kept = empty - free_bytes()
    assert kept > 64 << 20  # 16 x 16 x 256^2 fields and their tables
    ctx.set_option("pool_mb", 0)
    assert free_bytes() >= empty - (8 << 20)
    ctx.close()
