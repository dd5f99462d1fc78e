"""Matrix inverses of the chain on both sides of the four-wave kernel's range
(32 < n <= 48), through a chain with given matrices whose rows are permuted, so
that nearly every step pivots, against the oracle."""
import numpy as np
import pytest

import BoostFractor as B
from helpers import DISKR, O, chain_sensitivity, ocoords, rel
from test_gpu_transformer import _flat_booster, _lg_like_modes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 33, 41, 48, 49])
def test_chain_with_pivoting_inverses(n):
    coords, sb = _flat_booster(N=16, ndisk=2)
    modes = _lg_like_modes(coords, n, 0)
    rng = np.random.default_rng(n)
    mats = [np.eye(n, dtype=complex)]
    for _ in range(1, len(sb.distance)):
        x = np.eye(n) + 0.2 / np.sqrt(n) * (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
        mats.append(np.exp(2j * np.pi * rng.uniform(size=n))[:, None] * x[rng.permutation(n)])
    emit = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    got = B.transformer(sb.copy(), coords, modes, f=20e9, diskR=DISKR, emit=emit, propagation_matrices=mats)
    eps = sb.eps.copy()
    eps[np.isnan(eps.real)] = 1e30
    want = O.transformer(O.Setup(sb.distance, eps, None, sb.relative_tilt_x, sb.relative_tilt_y, None),
                         ocoords(coords), modes.patterns_flat()[:, 0], modes.mode_kt.reshape(-1), 20e9,
                         O.PROP_PROPAGATOR, prop_mats=mats, diskR=DISKR, emit=emit)
    tol = max(1e-10, 10 * chain_sensitivity(mats, eps, emit))
    assert tol < 1e-7 and rel(got, want) < tol, (rel(got, want), tol)
