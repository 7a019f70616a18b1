"""Where the plain form runs its chains: the plan of a shape, and both plans of
the shapes beside its lines against the oracle, bit for bit on integer
couplings."""

import ctypes
import os

import numpy as np
import pytest

import oracle
from pysa_amd import _lib
from helpers import (assert_same, engine_ais, engine_metropolis, int_problem, random_spins)

pytestmark = pytest.mark.gpu

READS, CHAINS = 0, 1


@pytest.fixture(scope="module")
def plan():
    ctypes.CDLL(_lib.load()._name, mode=ctypes.RTLD_GLOBAL)
    probe = ctypes.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_probe",
                                     "_build", "libhost_probe.so"))
    return lambda n, reads, R, S, dtype, coupled: probe.probe_plan_plain(
        n, reads, R, S, np.dtype(dtype).itemsize, int(coupled))


# The faster plan of each, measured on 256 compute units.
@pytest.mark.parametrize("n,reads,R,S,dtype,coupled,want", [
    # rounds of a read; short sweeps, short runs
    (16, 1, 17, 100, "f4", True, READS), (64, 8, 20, 100, "f4", True, READS),
    (50, 1, 20, 100, "f8", True, READS), (16, 1, 17, 2, "f4", True, CHAINS),
    (16, 1, 17, 100, "f4", False, CHAINS), (64, 1, 32, 100, "f4", True, CHAINS),
    (256, 1, 23, 100, "f4", True, CHAINS), (300, 1, 17, 100, "f4", True, CHAINS),
    (33, 130, 17, 100, "f4", True, READS),
    # long rows
    (2048, 1, 2, 9, "f4", True, CHAINS), (2048, 1, 1, 9, "f4", False, READS),
    (2048, 200, 2, 100, "f4", True, READS), (2500, 512, 1, 9, "f4", False, CHAINS),
    (4096, 1, 1, 9, "f4", False, CHAINS), (4096, 513, 1, 9, "f4", False, READS),
    # crowded compute units
    (50, 1, 16, 100, "f4", True, READS), (512, 1, 16, 100, "f4", True, READS),
    (512, 1, 16, 10, "f4", True, CHAINS), (1024, 1, 8, 100, "f4", True, READS),
    (1024, 1, 16, 100, "f4", True, CHAINS), (300, 8, 16, 100, "f8", True, CHAINS),
    (300, 32, 16, 100, "f8", True, CHAINS), (512, 1, 8, 100, "f8", True, READS),
    (1600, 128, 4, 100, "f8", True, READS), (1600, 64, 4, 100, "f8", True, CHAINS),
    (1024, 64, 8, 100, "f8", True, READS),
])
def test_plan(plan, n, reads, R, S, dtype, coupled, want):
    assert plan(n, reads, R, S, dtype, coupled) == want


def run(n, R, reads, S, dtype, ptype, order, best_sem=0, use_pt=True, log_omega=False):
    rng = np.random.default_rng([n, R, reads, order])
    J, h = int_problem(n, rng)
    J, h = J.astype(dtype), h.astype(dtype)
    betas = np.geomspace(1.0, 0.02, R).astype(dtype) if R > 1 else np.array([0.3], dtype)
    if log_omega:
        betas[-1] = 0.0
    st = random_spins((reads, R, n), rng, ptype)
    s = st.reshape(-1, n).astype(np.float64)
    en = (0.5 * np.sum((s @ J.astype(np.float64)) * s, axis=1) + s @ h.astype(np.float64))
    en = en.astype(dtype).reshape(reads, R)
    kw = dict(order=order, best_sem=best_sem, use_pt=use_pt, log_omega=log_omega, seed=3)
    want = oracle.metropolis(J, h, ptype, betas, st, en, S, nthreads=8, **kw)
    got = engine_metropolis(J, h, ptype, betas, st, en, S, **kw)
    assert_same(got, want)
    if log_omega:
        assert np.allclose(got["log_omegas"], want["log_omegas"], rtol=1e-12, atol=1e-12)


# A workgroup per read at the largest sizes: its replicas in registers (R = 1)
# and carried through memory (5 on 4 waves).
@pytest.mark.parametrize("n,R,reads,dtype", [(2100, 1, 520, "f4"), (2049, 5, 420, "f4"),
                                             (1100, 1, 300, "f8"), (1030, 5, 210, "f8")])
@pytest.mark.parametrize("ptype,order", [(0, 0), (1, 1)])
def test_large_reads(plan, n, R, reads, dtype, ptype, order):
    assert plan(n, reads, R, 1, dtype, R > 1) == READS
    run(n, R, reads, 1, np.dtype(dtype), ptype, order)


# Real couplings: the same chains in both plans (log-omega couples the sweeps and
# so takes the run to a workgroup per read, but changes nothing in the chains).
@pytest.mark.parametrize("n,R", [(16, 17), (64, 20), (130, 18), (255, 17)])
@pytest.mark.parametrize("dtype", ["f4", "f8"])
@pytest.mark.parametrize("ptype,order", [(0, 0), (0, 1), (1, 1), (1, 2), (1, 3)])
def test_plans_agree_on_real_couplings(plan, n, R, dtype, ptype, order):
    S = 131  # across a refresh in float32
    assert plan(n, 2, R, S, dtype, True) == READS and plan(n, 2, R, S, dtype, False) == CHAINS
    rng = np.random.default_rng([n, R, order])
    A = np.triu(rng.standard_normal((n, n)), 1) / np.sqrt(n)
    J, h = (A + A.T).astype(dtype), (0.1 * rng.standard_normal(n)).astype(dtype)
    betas = np.geomspace(3.0, 0.5, R).astype(dtype)
    betas[-1] = 0.0
    st = random_spins((2, R, n), rng, ptype)
    en = np.zeros((2, R), dtype)
    kw = dict(order=order, use_pt=False, seed=3)
    assert_same(engine_metropolis(J, h, ptype, betas, st, en, S, log_omega=True, **kw),
                engine_metropolis(J, h, ptype, betas, st, en, S, log_omega=False, **kw))


# Replicas carried through memory: ends of sweeps and, in float32, a refresh.
@pytest.mark.parametrize("dtype,reads,S", [("f4", 2, 131), ("f4", 130, 131), ("f8", 2, 16)])
@pytest.mark.parametrize("use_pt,best_sem,log_omega", [(True, 1, False), (True, 0, True),
                                                       (False, 1, False), (False, 0, True)])
def test_carried_replicas(plan, dtype, reads, S, use_pt, best_sem, log_omega):
    assert plan(70, reads, 17, S, dtype, True) == READS
    run(70, 17, reads, S, np.dtype(dtype), 0, 1, best_sem, use_pt, log_omega)


# More chains than the device takes one to a workgroup: waves side by side.
@pytest.mark.parametrize("n,dtype", [(300, "f4"), (1030, "f4"), (2100, "f4"), (600, "f8"), (1100, "f8")])
@pytest.mark.parametrize("ptype,order", [(0, 0), (1, 1)])
def test_many_ais_chains(n, dtype, ptype, order):
    rng = np.random.default_rng(n)
    J, h = int_problem(n, rng, -2, 2, 1)
    J, h = J.astype(dtype), h.astype(dtype)
    st = random_spins((515, n), rng, ptype)
    temps = np.array([0.05, 0.2], dtype)
    kw = dict(ref=1, p=0.4, order=order, seed=9)
    got, want = engine_ais(J, h, ptype, temps, st, **kw), oracle.ais(J, h, ptype, temps, st, **kw)
    assert np.array_equal(got[0], want[0])
    assert np.allclose(got[1], want[1], rtol=1e-12, atol=1e-10)
