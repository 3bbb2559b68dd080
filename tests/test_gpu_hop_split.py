"""The hopping kernels on either side of the lines between their forms (four,
two or one wave per site, operator kept in the caches or streamed), with site
counts that leave a remainder in the last workgroup.  Smaller lattices, which
the other tests use, all run the four-wave form.

FP64 against the oracle: a site's result is a sum of eight hops and a clover
product, each good to 1e-16 of its size, in another order than the oracle's;
bound 1e-13 of the largest value, as for the golden vectors (1e-12 after two
CG steps, whose scalars are sums over the lattice).  Reduced precision against
FP64 on the same device fields, with the bounds of the operator's own test."""
import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu
KAPPA, CSW, RHO = 0.125, 1.0, 0.07

# sites per parity: 35640 (two waves), 50400 (18-real links: one, kept; two-row: two),
# 131040 (18-real: one; two-row: two; both streamed), 146016 (one, streamed, in
# workgroups of one wave)
FP64 = [(10, 18, 22, 18), (14, 20, 12, 30), (26, 18, 20, 28), (26, 18, 24, 26)]
# 35640, 121680 (two waves, kept), 262080 (FP32: two, streamed), 554880 (one, streamed)
REDUCED = [(10, 18, 22, 18), (26, 18, 20, 26), (30, 26, 28, 24), (34, 30, 32, 34)]
TOL = {"f16": (1e-4, 3e-4), "f16g": (5e-5, 1e-4), "f32": (1e-6, 2e-6)}


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("L", FP64, ids=lambda L: "x".join(map(str, L)))
def test_fp64_operators(L):
    import bqcd_hip
    lat = ol.Lattice(L)
    u = lat.gauge_exp_random(31, 0.3)
    a, ai, b = lat.clover_init(u, CSW * KAPPA)
    flipped = lat.flip_bc(u)
    op = lat.op(flipped, a, ai, KAPPA, CSW * KAPPA, RHO)
    x = [lat.spinor_gauss(32, 0), lat.spinor_gauss(33, 1)]
    g = bqcd_hip.Lattice(L)
    g.load_gauge(u)
    g.load_clover(a, ai, b)
    for e in (0, 1):
        for dagger in (False, True):
            assert rel(g.d(e, x[1 - e], dagger), lat.d(e, int(dagger), x[1 - e], flipped)) < 1e-13, (e, dagger)
    assert rel(g.w_dagger_w(x[0], KAPPA, RHO), lat.apply(op, 5, x[0])) < 1e-13
    got, _, _ = g.cg("w_dagger_w", x[0], KAPPA, RHO, rest=0.0, maxiter=2, log=2)
    want, _, _ = lat.cg(op, 5, x[0], 0.0, 2)
    assert rel(got, want) < 1e-12
    g.close()


@pytest.mark.parametrize("L", REDUCED, ids=lambda L: "x".join(map(str, L)))
def test_reduced_operators(L):
    import torch
    import bqcd_hip
    g = bqcd_hip.Lattice(L)
    g.gauge_random(5, 0.3)
    g.build_clover(CSW * KAPPA)
    x = torch.empty((12, g.volh, 2), dtype=torch.float64, device="cuda")
    g.gaussian_d(x, 6, 0.5)
    y, z = torch.empty_like(x), torch.empty_like(x)
    for op in ("w_mult_dag", "w_dagger_w"):
        g.apply_d(op, KAPPA, RHO, y, x)
        for prec in ("f16", "f32", "f16g"):
            g.apply_lp_d(op, KAPPA, RHO, z, x, precision=prec)
            d = z - y
            worst = float(d.pow(2).sum(dim=(0, 2)).sqrt().max() / y.pow(2).sum(dim=(0, 2)).mean().sqrt())
            assert float(d.norm() / y.norm()) < TOL[prec][0] and worst < TOL[prec][1], (op, prec)
    g.close()
