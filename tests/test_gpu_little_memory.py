"""Solvers where little of the GPU's memory is left: they go without the further
search directions of their rings, which the same solve needs no memory for, and
end with the same numbers bit for bit (the same sums in the same order).  The
lattice is above every line from which search directions go round four buffers.
Memory is held by a tensor that is never touched; a fifth of it stays free."""
import pytest

pytestmark = pytest.mark.gpu
L, KAPPA, CSW = (26, 26, 28, 28), 0.12, 1.0


def solves(g, b):
    import torch
    bb = float(b.square().sum())
    bs = [b, b.roll(1, 1).contiguous(), -b]
    out = []
    x = torch.zeros_like(b)
    out += [x.clone(), g.cg_d("mtdagmt", x, b, KAPPA, rest=1e-10 * bb, maxiter=500), x]
    for prec in ("f32", "f16"):
        x = torch.zeros_like(b)
        out += [g.cg_mixed_d("mtdagmt", x, b, KAPPA, rest=1e-14 * bb, maxiter=500, precision=prec), x]
        xs = [torch.zeros_like(v) for v in bs]
        out += [g.cg_multi_d("mtdagmt", xs, bs, [KAPPA] * 3, csw=-1.0, rests=[1e-6 * bb, 1e-10 * bb, 1e-14 * bb],
                             maxiter=500, precision=prec, block=4), *xs]
    return out


def run(b):
    """results, and the device memory that the solves took"""
    import torch
    import bqcd_hip
    g = bqcd_hip.Lattice(L)
    g.gauge_random(11, 0.3)
    g.build_clover(CSW * KAPPA)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    out = solves(g, b)
    torch.cuda.synchronize()
    taken = before - torch.cuda.mem_get_info()[0]
    g.close()
    return out, taken


def test_solves_without_the_memory_of_a_ring():
    import torch
    import bqcd_hip
    g = bqcd_hip.Lattice(L)
    b = torch.empty((12, g.volh, 2), dtype=torch.float64, device="cuda")
    g.gaussian_d(b, 12, 0.5)
    spinor = 192 * g.volh
    g.close()
    keep = [torch.empty_like(b) for _ in range(60)]  # torch's pool holds the solves' tensors before the counting
    del keep
    roomy, taken = run(b)
    free, total = torch.cuda.mem_get_info()
    held = torch.empty(max(0, free - total // 5), dtype=torch.uint8, device="cuda")
    tight, taken_tight = run(b)
    del held
    torch.cuda.empty_cache()
    assert len(roomy) == len(tight)
    for u, v in zip(roomy, tight):
        assert torch.equal(u, v) if torch.is_tensor(u) else u == v
    assert taken - taken_tight > 3 * spinor
