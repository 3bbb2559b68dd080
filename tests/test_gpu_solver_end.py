"""Where a solve ends: the host enqueues one iteration beyond the last, which
must leave the solution, the counts and the state alone, whichever of the
state's two slots and of the search directions' four buffers the last
iteration ends in.  On both sides of the lines from which the search
directions go round four buffers (FP64 solves from 127 k sites per parity,
16-bit ones from 2^18).

The residual returned is |b - A x|^2 of the x returned, formed in FP64 by the
same operator: both are sums of 24 numbers per site of one size, in another
order, so 1e-10 of the sum is 1e4 times their rounding at 10^7 numbers.
Iteration counts are exact."""
import pytest

pytestmark = pytest.mark.gpu
KAPPA, CSW = 0.12, 1.0
LATTICES = [(4, 4, 6, 8), (26, 26, 28, 28)]


@pytest.fixture(scope="module", params=LATTICES, ids=lambda L: "x".join(map(str, L)))
def problem(request):
    import torch
    import bqcd_hip
    g = bqcd_hip.Lattice(request.param)
    g.gauge_random(11, 0.3)
    g.build_clover(CSW * KAPPA)
    b = torch.empty((12, g.volh, 2), dtype=torch.float64, device="cuda")
    g.gaussian_d(b, 12, 0.5)
    yield g, b
    g.close()


def residual(g, x, b):
    import torch
    ax = torch.empty_like(b)
    g.apply_d("mtdagmt", KAPPA, 0.0, ax, x)
    return float((b - ax).square().sum())


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9])
def test_end_at_maxiter(problem, n):
    import torch
    g, b = problem
    x = torch.zeros_like(b)
    it, rtr = g.cg_d("mtdagmt", x, b, KAPPA, rest=0.0, maxiter=n, log=2)
    assert it == n and abs(rtr - residual(g, x, b)) < 1e-10 * rtr
    for prec in ("f32", "f16", "f16g"):
        x.zero_()
        it, nrel, rtr = g.cg_mixed_d("mtdagmt", x, b, KAPPA, rest=0.0, maxiter=n, log=2, precision=prec)
        assert it == n and nrel >= 1 and abs(rtr - residual(g, x, b)) < 1e-10 * rtr, prec


def test_end_by_convergence_and_without_iterations(problem):
    import torch
    g, b = problem
    bb = float(b.square().sum())
    for prec in (None, "f32", "f16"):
        x = torch.zeros_like(b)
        for rest in (1e-6 * bb, 1e-16 * bb):  # the second solve starts from the first one's x
            if prec is None:
                _, rtr = g.cg_d("mtdagmt", x, b, KAPPA, rest=rest, maxiter=500)
                slack = 2.0  # stopped by the iterated residual
            else:
                _, _, rtr = g.cg_mixed_d("mtdagmt", x, b, KAPPA, rest=rest, maxiter=500, precision=prec)
                slack = 1.0 + 1e-6  # stopped by the true one; the bound is a float
            assert rtr <= slack * rest and abs(rtr - residual(g, x, b)) < 1e-6 * rtr, (prec, rest)
        if prec is not None:
            want = x.clone()
            it, _, _ = g.cg_mixed_d("mtdagmt", x, b, KAPPA, rest=1e-15 * bb, maxiter=500, precision=prec)
            assert it == 0 and torch.equal(x, want)


@pytest.mark.parametrize("prec", ["f32", "f16"])
@pytest.mark.parametrize("n", [1, 3, 4])
def test_right_hand_sides_that_end_apart(problem, prec, n):
    """each has its reliable updates and its end in iterations of its own, so
    that they start again from any of the four buffers; the residual returned
    is the true one, formed as above"""
    import torch
    g, b = problem
    bs = [b, b.roll(1, 1), b.roll(5, 1), -b.flip(0)][:n]
    bs = [v.contiguous() for v in bs]
    xs = [torch.zeros_like(v) for v in bs]
    rests = [float(v.square().sum()) * 10.0 ** -(5 + 3 * k) for k, v in enumerate(bs)]
    its, rtrs, _ = g.cg_multi_d("mtdagmt", xs, bs, [KAPPA] * n, csw=-1.0, rests=rests, maxiter=500,
                                precision=prec, block=1 if n == 1 else 4)
    assert its == sorted(its) and its[0] > 0
    for x, v, rest, rtr in zip(xs, bs, rests, rtrs):
        assert rtr <= (1.0 + 1e-6) * rest and abs(rtr - residual(g, x, v)) < 1e-6 * rtr
