"""Initial states drawn in one array are those of one NumPy call per read (or
chain), with the global RNG left in the same place."""

import numpy as np
import pytest

from pysa_amd import ais
from pysa_amd.sa import Solver


@pytest.mark.parametrize("ptype", ["ising", "qubo"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (2, 1030, 700)])
def test_random_spins_follow_the_per_read_draws(ptype, shape):
    solver = Solver(np.zeros((shape[2], shape[2])), ptype)
    np.random.seed(11)
    got = np.empty(shape, np.int8)
    solver._random_spins(got)
    after = np.random.random(3)
    np.random.seed(11)
    want = np.stack([np.random.randint(2, size=shape[1:]) for _ in range(shape[0])])
    if ptype == "ising":
        want = 2 * want - 1
    assert np.array_equal(got, want)
    assert np.array_equal(after, np.random.random(3))


@pytest.mark.parametrize("p", [0.5, 0.3, 0.999, 1e-4])
def test_bernoulli_rows_follow_the_element_draws(p):
    np.random.seed(5)
    want = np.stack([ais.bernoulli_prob_initialization(60, "qubo", (p,)) for _ in range(40)])
    after = np.random.random(3)
    np.random.seed(5)
    got = np.stack([np.random.binomial(1, 1 - p, size=60) for _ in range(40)])
    assert np.array_equal(got, want)
    assert np.array_equal(after, np.random.random(3))
