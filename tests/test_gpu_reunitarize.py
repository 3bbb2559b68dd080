"""The projection to SU(3) divides a column by its length: one rounding per
number.  Links n * 1 come back as exactly 1, since n / n is 1 for every n, while
a product with the rounded reciprocal is not (49 * (1 / 49) < 1)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["link update", "smearing"])
@pytest.mark.parametrize("n", [3.0, 49.0, 98.0, 103.0, 107.0])
def test_multiples_of_one_become_one(call, n):
    import bqcd_hip
    assert n * (1.0 / n) < 1.0 or n == 3.0
    g = bqcd_hip.Lattice((4, 2, 2, 4))
    one = np.zeros((4, 2, g.volh, 3, 3, 2))
    for k in range(3):
        one[..., k, k, 0] = 1.0
    g.load_gauge(n * one)
    if call == "smearing":
        g.gauge_smear(1, 0.0)  # (1 - alpha) U + alpha / 6 (staples), projected
    else:
        g.hmc_u(np.zeros((4, 2, g.volh, 8)), 0.1)
    assert np.array_equal(g.save_gauge(), one)
    g.close()
