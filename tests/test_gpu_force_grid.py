"""The forces on lattices that do not fill the force kernels' grid: fewer sites
than a wave, a remainder after the last full wave, workgroups left over after
the XCDs have shared out the time slices, and extents of two, where both
neighbours of a site are the same one.  Oracle: the C restatement.  A force is
a sum of some hundred products of unit-size numbers, each good to 1e-16, in
another order than the oracle's: 1e-13 of the largest value, as for the golden
vectors."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu
KAPPA, CSW, STEP, BETA = 0.125, 1.7, 0.37, 5.3
LATTICES = [(2, 2, 2, 2), (6, 4, 2, 4), (2, 10, 6, 4), (10, 6, 4, 14), (8, 8, 16, 6)]


@pytest.fixture(scope="module", params=LATTICES, ids=lambda L: "x".join(map(str, L)))
def case(request):
    import bqcd_hip
    lat = ol.Lattice(request.param)
    u = lat.gauge_exp_random(91, 0.4)
    a, ai, b = lat.clover_init(u, CSW * KAPPA)
    g = bqcd_hip.Lattice(request.param)
    g.load_gauge(u)
    g.load_clover(a, ai, b)
    yield g, lat, u, (a, ai, b)
    g.close()


def close(got, want):
    assert np.max(np.abs(got - want)) <= 1e-13 * np.max(np.abs(want))


def test_gauge_force(case):
    g, lat, u, _ = case
    close(g.dsg(STEP, BETA), lat.dsg(u, STEP, BETA))
