"""The pipelined MFMA kernel where its launch shapes change: two blocks, one or
two tiles per workgroup in every mode, and the two ways of its in-block field
updates (f32 MFMA with one tile, VALU with two)."""

import numpy as np
import pytest

import oracle
from pysa_amd import _lib
from helpers import (assert_same, energies_of, engine_ais, engine_metropolis, float_problem,
                     int_problem, random_spins)
from test_gpu_batched import compare, make_instances, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [33, 63, 64, 95])
@pytest.mark.parametrize("best_sem", [0, 1])
@pytest.mark.parametrize("kernel,tiles", [(1, 1), (1, 2), (2, 0), (0, 0)])
def test_two_and_three_blocks_with_log_omega(n, best_sem, kernel, tiles):
    rng = np.random.default_rng(n)
    J, h = int_problem(n, rng)
    J, h = J.astype(np.float32), h.astype(np.float32)
    R, reads, S = 16, 5, 25
    betas = np.append(np.geomspace(1.0, 0.05, R - 1), 0.0).astype(np.float32)
    st = random_spins((reads, R, n), rng, n & 1)
    en = energies_of(J, h, st, n & 1, np.float32)
    kw = dict(order=0, best_sem=best_sem, log_omega=True, seed=4)
    want = oracle.metropolis(J, h, n & 1, betas, st, en, S, **kw)
    prob = _lib.Problem(J, h, "ising" if n % 2 == 0 else "qubo", np.float32)
    prob.set_shape(kernel, tiles)
    got = engine_metropolis(J, h, n & 1, betas, st, en, S, form=_lib.FORM_BLOCKED, problem=prob,
                            **kw)
    prob.close()
    assert_same(got, want)
    assert np.allclose(got["log_omegas"], want["log_omegas"], rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("ptype", [0, 1])
@pytest.mark.parametrize("form", [_lib.FORM_BLOCKED, _lib.FORM_BLOCKED_EXACT])
@pytest.mark.parametrize("order", [0, 3])
def test_update_forms_round_alike(ptype, form, order):
    """Real couplings: every field of the f32 MFMA updates must round as the
    VALU's, or the chains part within a few sweeps (260 sweeps: past a
    recomputation of the energies)."""
    rng = np.random.default_rng(21 + ptype)
    n, R, reads, S = 203, 16, 3, 260
    J, h = float_problem(n, rng)
    J, h = J.astype(np.float32), h.astype(np.float32)
    betas = (1 / np.geomspace(0.1, 2.0, R)).astype(np.float32)
    st = random_spins((reads, R, n), rng, ptype)
    en = energies_of(J, h, st, ptype, np.float32)
    prob = _lib.Problem(J, h, "ising" if ptype == 0 else "qubo", np.float32)
    out = []
    for tiles in (1, 2):
        prob.set_shape(1, tiles)
        out.append(engine_metropolis(J, h, ptype, betas, st, en, S, order=order, seed=6, form=form,
                                     problem=prob))
    prob.close()
    assert_same(out[0], out[1])


@pytest.mark.parametrize("order", [0, 3])
@pytest.mark.parametrize("kind", ["int", "float"])
def test_ais_tiles(order, kind):
    """8200 chains run two tiles per workgroup, their first 100 alone one."""
    rng = np.random.default_rng(31)
    n = 70
    J, h = int_problem(n, rng) if kind == "int" else float_problem(n, rng)
    J, h = J.astype(np.float32), h.astype(np.float32)
    st = random_spins((8200, n), rng, 1)
    temps = np.linspace(0.0, 1.0, 5).astype(np.float32)
    kw = dict(order=order, seed=8, energies=True, form=_lib.FORM_BLOCKED)
    many = engine_ais(J, h, 1, temps, st, **kw)
    few = engine_ais(J, h, 1, temps, st[:100], **kw)
    for a, b in zip(many, few):
        assert np.array_equal(a[:100], b)


@pytest.mark.parametrize("count,reads,R", [(256, 1, 5), (257, 1, 5), (60, 9, 16)])
def test_batched_tiles(count, reads, R):
    """One tile per workgroup up to 256 tiles (a compute unit each), then two."""
    rng = np.random.default_rng(count)
    inst = make_instances(rng, rng.integers(65, 100, count), "int")
    for order in (0, 3):
        got, want, pk = run_both(inst, 0, reads, R, 4, order, 0, 5, True, rng, form="blocked")
        compare(got, want, pk, reads, R)
