"""Bernoulli initial states of annealed importance sampling: drawn row by row, they
are those of the reference's element draws, with the global RNG left in the same
place."""

import numpy as np
import pytest

from pysa_amd import ais
from pysa_amd.sa import Solver


@pytest.mark.parametrize("ptype", ["ising", "qubo"])
@pytest.mark.parametrize("p", [0.5, 0.3, 0.999, 1e-4])
@pytest.mark.parametrize("shape", [(1, 1), (40, 60)])
def test_solver_rows_follow_the_element_draws(ptype, p, shape):
    solver = Solver(np.zeros((shape[1], shape[1])), ptype)
    np.random.seed(5)
    want = np.stack([ais.bernoulli_prob_initialization(shape[1], ptype, (p,))
                     for _ in range(shape[0])])
    after = np.random.random(3)
    np.random.seed(5)
    got = np.empty(shape, np.int8)
    solver._bernoulli_spins(got, p)
    assert np.array_equal(got, want)
    assert np.array_equal(after, np.random.random(3))
