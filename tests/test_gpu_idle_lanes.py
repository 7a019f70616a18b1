"""Exchanges of the MFMA form with reads that leave lanes of a workgroup idle
behind a full ladder, against the oracle.  Whole-number couplings: equal bits."""

import numpy as np
import pytest

import oracle
from pysa_amd import _lib

from helpers import assert_same, energies_of, engine_metropolis, int_problem, random_spins

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,reads", [(12, 5), (24, 5), (43, 2), (60, 1)])
@pytest.mark.parametrize("best_sem", [0, 1])
def test_exchanges_beside_idle_lanes(R, reads, best_sem):
    n, S = 70, 12
    rng = np.random.default_rng(R)
    J, h = int_problem(n, rng, -3, 3, 2)
    J, h = J.astype(np.float32), h.astype(np.float32)
    betas = (1 / np.geomspace(3.0, 3.3, R)).astype(np.float32)
    st = random_spins((reads, R, n), rng, 0)
    en = energies_of(J, h, st, 0, np.float32)
    kw = dict(order=0, seed=5, best_sem=best_sem)
    assert_same(engine_metropolis(J, h, 0, betas, st, en, S, form=_lib.FORM_BLOCKED, **kw),
                oracle.metropolis(J, h, 0, betas, st, en, S, nthreads=8, **kw))
