"""The end of a sweep of the MFMA form against the oracle: exchange walks from
ladders that swap everything to ladders that swap nothing, one and several
reads per workgroup, and states whose length is no multiple of eight (stored
and loaded eight spins at a time).  Whole-number couplings: equal bits."""

import numpy as np
import pytest

import oracle
from pysa_amd import _lib

from helpers import assert_same, energies_of, engine_metropolis, int_problem, random_spins

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,reads", [(2, 17), (3, 11), (16, 5), (31, 3), (32, 3), (33, 2), (64, 2)])
@pytest.mark.parametrize("ladder", ["equal", "close", "wide"])
@pytest.mark.parametrize("best_sem", [0, 1])
def test_exchange_walks(R, reads, ladder, best_sem):
    n, S = 65 + R % 8, 12
    rng = np.random.default_rng(1000 + R)
    J, h = int_problem(n, rng, -3, 3, 2)
    J, h = J.astype(np.float32), h.astype(np.float32)
    top = {"equal": 3.0, "close": 3.3, "wide": 60.0}[ladder]
    betas = (1 / np.geomspace(3.0, top, R)).astype(np.float32)
    st = random_spins((reads, R, n), rng, 0)
    en = energies_of(J, h, st, 0, np.float32)
    ref = oracle.metropolis(J, h, 0, betas, st, en, S, order=0, seed=5, best_sem=best_sem, nthreads=8)
    got = engine_metropolis(J, h, 0, betas, st, en, S, order=0, seed=5, best_sem=best_sem,
                            form=_lib.FORM_BLOCKED)
    assert_same(got, ref)


@pytest.mark.parametrize("n", [65, 66, 71, 72, 95, 97, 111, 120, 127, 257])
@pytest.mark.parametrize("ptype", [0, 1])
@pytest.mark.parametrize("kind", ["int8", "bf16"])
def test_state_bytes(n, ptype, kind):
    rng = np.random.default_rng(2000 + n)
    lim = 3 if kind == "int8" else 200
    J, h = int_problem(n, rng, -lim, lim, 2)
    J, h = J.astype(np.float32), h.astype(np.float32)
    R, reads, S = 5, 3, 4
    betas = (1 / np.geomspace(float(lim), 30.0 * lim, R)).astype(np.float32)
    st = random_spins((reads, R, n), rng, ptype)
    en = energies_of(J, h, st, ptype, np.float32)
    ref = oracle.metropolis(J, h, ptype, betas, st, en, S, order=0, seed=5, nthreads=8)
    got = engine_metropolis(J, h, ptype, betas, st, en, S, order=0, seed=5, form=_lib.FORM_BLOCKED)
    assert_same(got, ref)
