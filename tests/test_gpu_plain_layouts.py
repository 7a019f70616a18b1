"""The plain form in both of its layouts (one workgroup per read, one per
chain) against the oracle, bit for bit on integer couplings, at the edges of
its 64-visit windows and 256-element row chunks."""

import numpy as np
import pytest

import oracle
from helpers import (assert_same, energies_of, engine_ais, engine_metropolis, int_problem,
                     random_spins, replay_arrays)

pytestmark = pytest.mark.gpu


def run(n, R, reads, S, dtype, ptype, order, best_sem=0, use_pt=True, log_omega=False, seed=3):
    rng = np.random.default_rng([n, R, reads, order])
    J, h = int_problem(n, rng)
    J, h = J.astype(dtype), h.astype(dtype)
    betas = np.geomspace(1.0, 0.02, R).astype(dtype) if R > 1 else np.array([0.3], dtype)
    if log_omega:
        betas[-1] = 0.0
    st = random_spins((reads, R, n), rng, ptype)
    en = energies_of(J, h, st, ptype, dtype)
    kw = dict(order=order, best_sem=best_sem, use_pt=use_pt, log_omega=log_omega, seed=seed)
    want = oracle.metropolis(J, h, ptype, betas, st, en, S, **kw)
    got = engine_metropolis(J, h, ptype, betas, st, en, S, **kw)
    assert_same(got, want)
    if log_omega:
        assert np.allclose(got["log_omegas"], want["log_omegas"], rtol=1e-12, atol=1e-12)


# (R, reads): 33 replicas go to one workgroup per chain, 5 to one per read
@pytest.mark.parametrize("R,reads", [(33, 2), (5, 3)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("order", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 31, 63, 65, 255, 257, 513, 1030])
def test_edges(n, order, dtype, R, reads):
    run(n, R, reads, 3, dtype, n & 1, order)


@pytest.mark.parametrize("R,reads", [(40, 1), (1, 3), (16, 2)])
@pytest.mark.parametrize("use_pt,best_sem,log_omega", [(True, 1, False), (False, 0, False),
                                                       (False, 1, False), (True, 0, True),
                                                       (False, 0, True)])
def test_ends_of_sweeps_across_a_refresh(use_pt, best_sem, log_omega, R, reads):
    if log_omega and R == 1:
        pytest.skip("log-omega needs a ladder")
    run(70, R, reads, 131, np.float32, 0, 1, best_sem, use_pt, log_omega)


def test_largest_sizes():
    run(3000, 20, 1, 2, np.float32, 0, 0)  # 12 of 16 row chunks
    run(4096, 3, 1, 1, np.float32, 1, 1)
    run(2048, 5, 1, 1, np.float64, 0, 1)
    run(1300, 5, 1, 1, np.float64, 0, 0)  # 6 of 8


@pytest.mark.parametrize("R,reads", [(1000, 1), (17, 130)])
def test_many_replicas(R, reads):
    run(33, R, reads, 3, np.float32, 0, 1)


@pytest.mark.parametrize("R", [3, 20])
def test_replayed_order_that_repeats_positions(R):
    """The reference visits whatever positions it is given, one after another."""
    rng = np.random.default_rng(R)
    n, reads, S = 100, 2, 3
    J, h = int_problem(n, rng)
    J, h = J.astype(np.float32), h.astype(np.float32)
    betas = np.geomspace(0.5, 0.05, R).astype(np.float32)
    st = random_spins((reads, R, n), rng, 0)
    en = energies_of(J, h, st, 0, np.float32)
    rep = replay_arrays(rng, reads, S, R, n, random_order=True)
    rep["perm"] = rng.integers(0, n, rep["perm"].shape).astype(np.int32)
    kw = dict(order=1, replay=rep)
    assert_same(engine_metropolis(J, h, 0, betas, st, en, S, **kw),
                oracle.metropolis(J, h, 0, betas, st, en, S, **kw))


# a workgroup per chain up to 512 chains, then waves spread over the device
@pytest.mark.parametrize("chains", [2, 512, 513, 1100])
@pytest.mark.parametrize("n,order", [(40, 1), (65, 0), (300, 1)])
def test_ais_layouts(chains, n, order):
    rng = np.random.default_rng(chains + n)
    J, h = int_problem(n, rng, -2, 2, 1)
    J, h = J.astype(np.float64), h.astype(np.float64)
    st = random_spins((chains, n), rng, 1)
    temps = np.array([0.05, 0.1, 0.2])
    for ref in (0, 1):
        kw = dict(ref=ref, p=0.4, order=order, seed=9)
        got, want = engine_ais(J, h, 1, temps, st, **kw), oracle.ais(J, h, 1, temps, st, **kw)
        assert np.array_equal(got[0], want[0])
        assert np.allclose(got[1], want[1], rtol=1e-12, atol=1e-10)
