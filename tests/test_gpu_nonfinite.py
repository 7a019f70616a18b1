"""Infinite couplings: an unset QUBO spin adds nothing to a field, whichever way
the chains run, so the per-read and the per-chain plan answer alike, and both
like the sparse form (always per read); without unset spins, like the oracle."""

import numpy as np
import pytest

import oracle
from pysa_amd import _lib
from helpers import engine_metropolis, int_problem, random_spins

pytestmark = pytest.mark.gpu


# 5 replicas run in a workgroup per read, 40 one to a workgroup
@pytest.mark.parametrize("n", [40, 300])
@pytest.mark.parametrize("R,reads", [(5, 2), (40, 1)])
@pytest.mark.parametrize("ptype", [0, 1])
@pytest.mark.parametrize("value", [np.inf, -np.inf])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_infinite_couplings(n, R, reads, ptype, value, dtype):
    rng = np.random.default_rng(n)
    J, h = int_problem(n, rng)
    J, h = J.astype(dtype), h.astype(dtype)
    J *= np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= 3
    J[3, 7] = J[7, 3] = value
    betas = np.geomspace(1.0, 0.02, R).astype(dtype)
    st = random_spins((reads, R, n), rng, ptype)
    en = np.zeros((reads, R), dtype)
    kw = dict(order=1, seed=3)
    got = engine_metropolis(J, h, ptype, betas, st, en, 3, form=_lib.FORM_PLAIN, **kw)
    wants = [engine_metropolis(J, h, ptype, betas, st, en, 3, form=_lib.FORM_SPARSE, **kw)]
    if ptype == 0:
        wants.append(oracle.metropolis(J, h, ptype, betas, st, en, 3, **kw))
    for want in wants:
        for k in ("states", "beta_idx", "best_state", "best_sweeps", "accepted"):
            assert np.array_equal(got[k], want[k]), k
        for k in ("energies", "best_energy"):
            assert np.array_equal(got[k], want[k], equal_nan=True), k
