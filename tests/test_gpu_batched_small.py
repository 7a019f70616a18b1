"""Batches of at most 64 spins (one window of visits, couplings in LDS) and the
general plain kernel around its 64-visit windows, against the batched oracle."""

import numpy as np
import pytest

from test_gpu_batched import compare, make_instances, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1, 2, 31, 32, 33, 63, 64], [64, 65, 127, 129, 257]])
@pytest.mark.parametrize("order", [0, 1, 2, 3])
@pytest.mark.parametrize("R,reads,best_sem", [(1, 3, 0), (16, 2, 1), (5, 2, 0)])
def test_batched_windows(sizes, order, R, reads, best_sem):
    rng = np.random.default_rng(7 * R + order)
    inst = make_instances(rng, sizes, "int")
    got, want, pk = run_both(inst, order & 1, reads, R, 6, order, best_sem, 3, True, rng)
    compare(got, want, pk, reads, R)
