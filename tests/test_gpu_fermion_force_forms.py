"""The fermion force on lattices of the further forms of its operator (D with the
LDL^+ solve behind it): two waves per site, and one wave with the operator kept in
the caches, streamed, and in workgroups of one wave.  The other force tests stay
below 33 k sites per parity, where four waves share a site.  Oracle and bound
(1e-13 of the largest value) as in the test of the force kernels' grid."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu
KAPPA, CSW, STEP = 0.125, 1.7, 0.37
# 35640, 50400, 131040 and 146016 sites per parity
LATTICES = [(10, 18, 22, 18), (14, 20, 12, 30), (26, 18, 20, 28), (26, 18, 24, 26)]


@pytest.mark.parametrize("L", LATTICES, ids=lambda L: "x".join(map(str, L)))
def test_fermion_force(L):
    import bqcd_hip
    lat = ol.Lattice(L)
    u = lat.gauge_exp_random(91, 0.4)
    a, ai, b = lat.clover_init(u, CSW * KAPPA)
    x, y = lat.spinor_gauss(6, 0), lat.spinor_gauss(7, 0)
    flipped = lat.flip_bc(u)
    want = lat.dsf(lat.op(flipped, a, ai, KAPPA, CSW * KAPPA), flipped, STEP, x, y, b)
    g = bqcd_hip.Lattice(L)
    g.load_gauge(u)
    g.load_clover(a, ai, b)
    got = g.dsf(x, y, STEP, KAPPA, CSW * KAPPA)
    g.close()
    assert float(np.max(np.abs(got - want))) <= 1e-13 * float(np.max(np.abs(want)))
