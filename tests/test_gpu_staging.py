"""Host-pointer calls of changing sizes on one problem (its kept staging memory
grows, holds smaller calls, and steps between the pinned and the direct
copies) give what a fresh problem gives."""

import numpy as np
import pytest

from pysa_amd import _lib
from helpers import assert_same, energies_of, engine_metropolis, int_problem, random_spins

pytestmark = pytest.mark.gpu


def test_one_problem_many_sizes():
    rng = np.random.default_rng(2)
    n = 130
    J, h = int_problem(n, rng)
    J, h = J.astype(np.float32), h.astype(np.float32)
    kept = _lib.Problem(J, h, "ising", np.float32)
    # 8 KB, just above and below 1 MiB, 4 MB, then small again
    for reads, R in ((2, 8), (1030, 8), (900, 8), (1000, 32), (1, 3)):
        betas = np.geomspace(1.0, 0.1, R).astype(np.float32)
        st = random_spins((reads, R, n), rng, 0)
        en = energies_of(J, h, st, 0, np.float32)
        assert np.array_equal(kept.energy(st.reshape(-1, n)), en.reshape(-1))
        for form, order, log_omega in ((_lib.FORM_PLAIN, 1, False), (_lib.FORM_BLOCKED, 3, False)):
            kw = dict(order=order, seed=reads, form=form, log_omega=log_omega)
            a = engine_metropolis(J, h, 0, betas, st, en, 3, problem=kept, **kw)
            b = engine_metropolis(J, h, 0, betas, st, en, 3, **kw)
            assert_same(a, b)
    kept.close()
