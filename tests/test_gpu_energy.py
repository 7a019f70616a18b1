"""The f64 energy kernel at the edges of its tilings: 4 states x 256 elements
below 4096 states (sums in a second launch above 256 spins), 16 states x 1024
elements from there, spins of any int8 value on both."""

import numpy as np
import pytest

from pysa_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("values", ["pm1", "01", "any"])
@pytest.mark.parametrize("n,count", [(1, 1), (63, 5), (256, 3), (257, 9), (1100, 4), (33, 4095),
                                     (65, 4096), (257, 4099), (1027, 4100)])
def test_energy_is_the_f64_sum(n, count, values, dtype):
    rng = np.random.default_rng(n + count)
    A = np.triu(rng.integers(-9, 10, (n, n)), 1)
    J = (A + A.T).astype(dtype)
    h = rng.integers(-5, 6, n).astype(dtype)
    if values == "any":
        st = rng.integers(-3, 4, (count, n)).astype(np.int8)
        st[0] = 1  # a group of states may hold both kinds
    else:
        b = rng.integers(0, 2, (count, n))
        st = (2 * b - 1 if values == "pm1" else b).astype(np.int8)
    prob = _lib.Problem(J, h, "ising", dtype)
    s = st.astype(np.float64)
    want = 0.5 * np.sum((s @ J.astype(np.float64)) * s, axis=1) + s @ h.astype(np.float64)
    # whole numbers (and halves) below 2^53: every order of the sums is exact
    assert np.array_equal(prob.energy(st), want)
    prob.close()


def test_energy_of_real_couplings_in_both_tilings():
    """The same states through either tiling: the sums run in the same order,
    so the values agree to the bit; f64 numpy to its own rounding."""
    rng = np.random.default_rng(5)
    n = 700
    A = np.triu(rng.standard_normal((n, n)), 1)
    J = (A + A.T).astype(np.float32)
    h = rng.standard_normal(n).astype(np.float32)
    st = (2 * rng.integers(0, 2, (4096, n)) - 1).astype(np.int8)
    prob = _lib.Problem(J, h, "ising", np.float32)
    wide = prob.energy(st)
    narrow = np.concatenate([prob.energy(st[:100]), prob.energy(st[100:])])
    assert np.array_equal(wide, narrow)
    s = st.astype(np.float64)
    want = 0.5 * np.sum((s @ J.astype(np.float64)) * s, axis=1) + s @ h.astype(np.float64)
    # sums of n^2 terms of magnitude ~1: n rounding steps of 2^-53 each on partial sums < n
    assert np.max(np.abs(wide - want)) < n * n * 2.0**-53 * 4
    prob.close()
