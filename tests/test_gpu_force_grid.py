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


def test_fermion_force(case):
    g, lat, u, (a, ai, b) = case
    x, y = lat.spinor_gauss(6, 0), lat.spinor_gauss(7, 0)
    flipped = lat.flip_bc(u)
    want = lat.dsf(lat.op(flipped, a, ai, KAPPA, CSW * KAPPA), flipped, STEP, x, y, b)
    close(g.dsf(x, y, STEP, KAPPA, CSW * KAPPA), want)


def test_clover_determinant_force(case):
    g, lat, u, (a, ai, b) = case
    close(g.dsd(STEP, CSW * KAPPA), lat.dsd(b, STEP, CSW * KAPPA, u))


def shifted(lat, f, eo_axis, site_axis):
    """a field moved by one site in t: the parities swap and the site index, whose
    slowest coordinate is t, moves by one slice"""
    return np.ascontiguousarray(np.roll(np.flip(f, eo_axis), lat.volh // lat.L[3], site_axis))


def test_one_parity(case):
    """clover_dsf and clover_dsd of one parity: even spinors against dsf at kappa = 0
    (no hopping and no odd part), odd factors against dsd; the other parities
    against these on fields moved by one site"""
    import bqcd_hip
    g, lat, u, (a, ai, b) = case
    x, y = lat.spinor_gauss(8, 0), lat.spinor_gauss(9, 0)
    ck = CSW * KAPPA
    s = -STEP * 2.0 * ck / 8.0
    even, odd = lat.gen(), lat.gen()
    g.clover_dsf(0, even, y, x, s)
    close(even, lat.dsf(lat.op(u, a, ai, 0.0, ck), u, STEP, x, y, b))
    g.clover_dsd(1, odd, s)
    close(odd, lat.dsd(b, STEP, ck, u))
    moved = bqcd_hip.Lattice(lat.L)
    moved.load_gauge(shifted(lat, u, 1, 2))
    moved.load_clover(*[shifted(lat, f, 0, 1) for f in (a, ai, b)])
    p, q = lat.gen(), lat.gen()
    n = lat.volh // lat.L[3]
    moved.clover_dsf(1, p, np.roll(y, n, 0), np.roll(x, n, 0), s)
    close(p, shifted(lat, even, 1, 2))
    moved.clover_dsd(0, q, s)
    close(q, shifted(lat, odd, 1, 2))
    moved.close()
