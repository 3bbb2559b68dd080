"""The solution a solver holds after n iterations, against a conjugate gradient
written here in torch on the FP64 operator.  A search direction that the ring of
a solver loses, adds twice or takes from the wrong slot changes x by a whole
step, which no residual recomputed from that x would show; the tolerances are
below a fifth of the last step (asserted), so that each such change fails.

On the lattices that separate the forms of the vector updates: 720 sites per
parity (workgroups of one wave, a remainder), 75816 (16-bit updates in workgroups
of four waves), 148720 (FP64 directions in a ring; more than 2048 partial sums
of <p, Ap>) and 265k (16-bit directions in a ring, sums in launches of their own).

Tolerances: FP64 sums over the lattice are good to 1e-14 and a condition number
of 1e2 to 1e3 multiplies that; FP32 fields are good to 6e-8, 16-bit links, clover and
spinors to 3e-5 of a site's largest number, multiplied likewise on the smooth
part of x: 1e-11, 1e-5 and 2e-3 of |x|."""
import pytest

pytestmark = pytest.mark.gpu
KAPPA, CSW = 0.13, 1.0
LATTICES = [(6, 4, 10, 6), (26, 18, 18, 18), (26, 26, 20, 22), (26, 26, 28, 28)]
TOL = {"f64": 1e-11, "f32": 1e-5, "f16": 2e-3, "f16g": 2e-3}
N = 9


def iterates(g, x0, b):
    """x after 0, 1, .. N iterations of the CG on M~^+ M~ from x0"""
    import torch
    ap = torch.empty_like(b)
    g.apply_d("mtdagmt", KAPPA, 0.0, ap, x0)
    r = b - ap
    p, x, rr = r.clone(), x0.clone(), r.square().sum()
    out = [x.clone()]
    for _ in range(N):
        g.apply_d("mtdagmt", KAPPA, 0.0, ap, p)
        alpha = rr / (p * ap).sum()
        x = x + alpha * p
        r = r - alpha * ap
        new = r.square().sum()
        p = r + (new / rr) * p
        rr = new
        out.append(x)
    return out


@pytest.fixture(scope="module", params=LATTICES, ids=lambda L: "x".join(map(str, L)))
def problem(request):
    import torch
    import bqcd_hip
    g = bqcd_hip.Lattice(request.param)
    g.gauge_random(11, 0.3)
    g.build_clover(CSW * KAPPA)
    bs = []
    for seed in (12, 13, 14):
        b = torch.empty((12, g.volh, 2), dtype=torch.float64, device="cuda")
        g.gaussian_d(b, seed, 0.5)
        bs.append(b)
    x0 = [0.02 * b.roll(1, 1) for b in bs]
    want = [iterates(g, x, b) for x, b in zip(x0, bs)]
    yield g, bs, x0, want
    g.close()


def compare(x, want, n, prec):
    size = float(want[n].norm())
    assert float((want[n] - want[n - 1]).norm()) > 5.0 * TOL[prec] * size
    assert float((x - want[n]).norm()) < TOL[prec] * size, (prec, n)


@pytest.mark.parametrize("n", range(1, N + 1))
def test_x_after_n_iterations(problem, n):
    g, bs, x0, want = problem
    x = x0[0].clone()
    it, _ = g.cg_d("mtdagmt", x, bs[0], KAPPA, rest=0.0, maxiter=n, log=2)
    assert it == n
    compare(x, want[0], n, "f64")
    for prec in ("f32", "f16", "f16g"):
        for delta in (0.1, 1e-9):  # with reliable updates on the way, and with none before the end
            x = x0[0].clone()
            it, nrel, _ = g.cg_mixed_d("mtdagmt", x, bs[0], KAPPA, rest=0.0, maxiter=n, log=2, precision=prec,
                                       delta=delta)
            assert it == n and (nrel == 1 or delta == 0.1)
            compare(x, want[0], n, prec)


@pytest.mark.parametrize("block", [1, 2, 4])
@pytest.mark.parametrize("prec", ["f32", "f16"])
def test_x_after_n_iterations_of_a_block(problem, prec, block):
    g, bs, x0, want = problem
    for n in range(1, N + 1):
        xs = [x.clone() for x in x0]
        its, _, _ = g.cg_multi_d("mtdagmt", xs, bs, [KAPPA] * 3, csw=-1.0, rests=[0.0] * 3, maxiter=n, log=2,
                                 precision=prec, block=block)
        assert its == [n] * 3
        for x, w in zip(xs, want):
            compare(x, w, n, prec)


def test_iteration_counts(problem):
    """a direction missing from x costs iterations at the next reliable update:
    FP32 solves take no more than a fifth above the FP64 solve's, 16-bit ones
    no more than twice"""
    import torch
    g, bs, _, _ = problem
    rests = [float(b.square().sum()) * rel for b, rel in zip(bs, (1e-7, 1e-11, 1e-15))]
    count = [g.cg_d("mtdagmt", torch.zeros_like(b), b, KAPPA, rest=rest, maxiter=500)[0]
             for b, rest in zip(bs, rests)]
    assert count == sorted(count) and count[0] > N
    for prec, most in (("f32", 1.2), ("f16", 2.0), ("f16g", 2.0)):
        its = [g.cg_mixed_d("mtdagmt", torch.zeros_like(b), b, KAPPA, rest=rest, maxiter=500, precision=prec)[0]
               for b, rest in zip(bs, rests)]
        assert all(i <= most * c + 2 for i, c in zip(its, count)), (prec, its, count)
        if prec == "f16g":
            continue
        for block in (1, 4):
            its, _, _ = g.cg_multi_d("mtdagmt", [torch.zeros_like(b) for b in bs], bs, [KAPPA] * 3, csw=-1.0,
                                     rests=rests, maxiter=500, precision=prec, block=block)
            assert all(i <= most * c + 2 for i, c in zip(its, count)), (prec, block, its, count)
