"""The f64 workspaces of the plain form and of the energies hold a bounded number
of states at a time: results equal those of one piece (oracle, NumPy), and what
a problem keeps behind a large call stays small."""

import numpy as np
import pytest
import torch

import oracle
from pysa_amd import _lib
from helpers import assert_same, engine_metropolis, int_problem, random_spins

pytestmark = pytest.mark.gpu


def problem(n, dtype=np.float32):
    rng = np.random.default_rng(n)
    J, h = int_problem(n, rng)
    return rng, J.astype(dtype), h.astype(dtype)


def energies_of(J, h, states):
    """f64 energies by matrix products (exact for these whole numbers)."""
    s = states.reshape(-1, states.shape[-1]).astype(np.float64)
    e = 0.5 * np.sum((s @ J.astype(np.float64)) * s, axis=1) + s @ h.astype(np.float64)
    return e.reshape(states.shape[:-1])


# 16 MB of 8 bytes: 2036 chains of 1030 spins
@pytest.mark.parametrize("ptype", [0, 1])
@pytest.mark.parametrize("reads", [2, 3])  # one piece, two with a ragged last group of four
def test_chains_in_pieces(ptype, reads):
    n, R, S = 1030, 1001, 1
    rng, J, h = problem(n)
    betas = np.geomspace(1.0, 0.02, R).astype(np.float32)
    st = random_spins((reads, R, n), rng, ptype)
    en = energies_of(J, h, st).astype(np.float32)
    kw = dict(order=1, seed=3)
    assert_same(engine_metropolis(J, h, ptype, betas, st, en, S, **kw),
                oracle.metropolis(J, h, ptype, betas, st, en, S, nthreads=8, **kw))


@pytest.mark.parametrize("count", [1904, 1905, 4001])  # 1904 of 1100 spins to a piece
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_energies_in_pieces(count, dtype):
    rng, J, h = problem(1100, dtype)
    s = random_spins((count, 1100), rng, count & 1)
    prob = _lib.Problem(J, h, "ising", dtype)
    assert np.array_equal(prob.energy(s), energies_of(J, h, s))
    prob.close()


def test_little_kept_behind_many_energies():
    n, count = 3000, 4000
    rng, J, h = problem(n)
    s = random_spins((count, n), rng, 0)
    prob = _lib.Problem(J, h, "ising", np.float32)
    prob.energy(s[:1])
    before = torch.cuda.mem_get_info()[0]
    prob.energy(s)
    kept = before - torch.cuda.mem_get_info()[0]
    prob.close()
    assert kept <= 64 << 20  # the states' 12 MB and a workspace of 16; 96 + 12 in one piece
