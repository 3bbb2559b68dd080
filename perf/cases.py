"""Timed cases of the BQCD hot path: the calls a lattice-QCD program makes, over
the range of lattices, precisions and options they are made with.

A case is a dict with a "kind" (which call), a lattice "L" ("XxYxZxT") and the
call's options.  listed() gives the fixed cases, draw(rng) another one of the
same ranges, prepare(case, seed) the inputs and the Lattice a program holds
before the call, run(state) one pass, work(case) the bytes and operations the
pass cannot do without, and exact(case, seed) the result of the same inputs in
plain torch FP64 arithmetic.

Links are Haar-random SU(3) matrices smoothed by five APE sweeps (plaquette
about 0.55), the benchmark's field; spinors and momenta are Gaussian.  Time is
antiperiodic for the fermions.
"""
import math
import os
import sys

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(REPO, "bqcd-r399-quda_amd"))

import bqcd_hip  # noqa: E402

CSW = 1.9
BETA = 5.29
RHO = 0.1
STEP = 0.025       # molecular-dynamics step of the link update and the kicks
HOP_FLOPS = 1320   # hopping term per output site
CLOVER_FLOPS = 504


def listed():
    return [
        # one hopping term on a lattice so small that the launch is all there is
        {"name": "dslash-6x4x10x8", "kind": "dslash", "L": "6x4x10x8", "parity": 1, "dagger": True},
        # the even-odd operator on the benchmark's lattice: bandwidth
        {"name": "mtdagmt-32x32x32x64", "kind": "apply", "L": "32x32x32x64", "op": "mtdagmt", "kappa": 0.1355},
        # the Hasenbusch-shifted operator on a lattice with no power of two in it
        {"name": "wdagw-20x12x10x36", "kind": "apply", "L": "20x12x10x36", "op": "w_dagger_w", "kappa": 0.13},
        # the plain FP64 solve on the 8^4 configuration: latency of an iteration
        {"name": "cg-8x8x8x8", "kind": "cg", "L": "8x8x8x8", "op": "mtdagmt", "kappa": 0.13},
        # the same, the drop-in for BQCD's cg(), on the smp benchmark input's lattice
        {"name": "cg-24x24x24x48", "kind": "cg", "L": "24x24x24x48", "op": "mtdagmt", "kappa": 0.13},
        # a mixed-precision solve of W^+W with FP32 storage, ragged lattice
        {"name": "mixed32-14x20x12x30", "kind": "mixed", "L": "14x20x12x30", "op": "w_dagger_w", "kappa": 0.13,
         "precision": "f32"},
        # the benchmark's solve: 16-bit storage, 32^3x64, at a quark mass where every
        # random field converges (near 0.1355 some have an almost zero mode)
        {"name": "mixed16-32x32x32x64", "kind": "mixed", "L": "32x32x32x64", "op": "mtdagmt", "kappa": 0.133,
         "precision": "f16"},
        # the batched solve: 12 right-hand sides over three quark masses
        {"name": "multi12-24x24x24x48", "kind": "multi", "L": "24x24x24x48", "nrhs": 12, "masses": 3,
         "kappa": 0.133, "precision": "f16"},
        # fermion force of the differentiation configuration
        {"name": "dsf-16x16x16x32", "kind": "dsf", "L": "16x16x16x32", "kappa": 0.135},
        # Wilson gauge force on the benchmark's lattice: the most frequent force of a trajectory
        {"name": "dsg-32x32x32x64", "kind": "dsg", "L": "32x32x32x64"},
        # one molecular-dynamics step without its solve: link update, clover
        # rebuild, all three forces, on a ragged lattice
        {"name": "md-24x20x12x36", "kind": "md", "L": "24x20x12x36", "kappa": 0.135},
        # a short trajectory with the 16-bit solver, and the links it ends with
        {"name": "hmc-12x12x12x24", "kind": "hmc", "L": "12x12x12x24", "kappa": 0.13, "precision": "f16"},
    ]


# sites of the smallest and largest lattice each kind is drawn with
SIZES = {"dslash": (1 << 11, 1 << 21), "apply": (1 << 11, 1 << 21), "cg": (1 << 11, 1 << 19),
         "mixed": (1 << 13, 1 << 20), "multi": (1 << 13, 1 << 18), "dsf": (1 << 11, 1 << 19),
         "dsg": (1 << 11, 1 << 21), "md": (1 << 11, 1 << 18), "hmc": (1 << 11, 1 << 15)}


def draw(rng):
    kind = rng.choice(sorted(SIZES))
    lo, hi = SIZES[kind]
    want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    while True:
        # even extents around the fourth root of the volume, time longer
        r = [math.exp(rng.uniform(-0.5, 0.5)) for _ in range(3)]
        side = (want / 2.0) ** 0.25
        L = [max(4, 2 * round(side * f / 2)) for f in r]
        L.append(max(4, 2 * round(want / (2 * L[0] * L[1] * L[2]))))
        if lo <= L[0] * L[1] * L[2] * L[3] <= hi and L[3] <= 96:
            break
    case = {"kind": kind, "L": "x".join(str(n) for n in L)}
    kappa = round(rng.uniform(0.12, 0.133), 4)
    if kind == "dslash":
        case.update(parity=rng.randrange(2), dagger=rng.random() < 0.5)
    elif kind == "apply":
        case.update(op=rng.choice(sorted(bqcd_hip.OP)), kappa=kappa)
    elif kind == "cg":
        case.update(op=rng.choice(["mtdagmt", "w_dagger_w"]), kappa=kappa)
    elif kind == "mixed":
        case.update(op=rng.choice(["mtdagmt", "w_dagger_w"]), kappa=kappa, precision=rng.choice(["f32", "f16"]))
    elif kind == "multi":
        case.update(nrhs=rng.randint(2, 12), masses=rng.randint(1, 2), kappa=kappa,
                    precision=rng.choice(["f32", "f16", "f16"]))
    elif kind in ("dsf", "md"):
        case.update(kappa=kappa)
    elif kind == "hmc":
        case.update(kappa=kappa, precision=rng.choice(["f64", "f32", "f16"]))
    return case


def extents(case):
    return tuple(int(n) for n in case["L"].split("x"))


def sites_per_parity(case):
    x, y, z, t = extents(case)
    return x * y * z * t // 2


# ---------------------------------------------------------------------------
# fields in plain torch: complex128, site index s = parity * volh + i with the
# even-odd order i = (x + LX (y + LY (z + LZ t))) / 2
# ---------------------------------------------------------------------------
DEV = "cuda"


class Grid:
    """neighbour tables and boundary signs of a lattice"""

    def __init__(self, L):
        self.L, self.volh = L, L[0] * L[1] * L[2] * L[3] // 2
        i = torch.arange(self.volh, device=DEV)
        xh, r = i % (L[0] // 2), i // (L[0] // 2)
        y, r = r % L[1], r // L[1]
        z, t = r % L[2], r // L[2]
        pos = []
        for eo in range(2):
            pos.append(torch.stack([2 * xh + (y + z + t + eo) % 2, y, z, t]))
        self.x = torch.cat(pos, 1)  # (4, 2 volh)
        self.fwd = [self.index(mu, 1) for mu in range(4)]
        self.bwd = [self.index(mu, -1) for mu in range(4)]
        one = torch.ones(2 * self.volh, device=DEV, dtype=torch.float64)
        self.fsign = [one] * 3 + [torch.where(self.x[3] == L[3] - 1, -one, one)]
        self.bsign = [one] * 3 + [torch.where(self.x[3] == 0, -one, one)]

    def index(self, mu, d):
        c = [self.x[k] for k in range(4)]
        c[mu] = (c[mu] + d) % self.L[mu]
        L = self.L
        lex = c[0] + L[0] * (c[1] + L[1] * (c[2] + L[2] * c[3]))
        return ((c[0] + c[1] + c[2] + c[3]) % 2) * self.volh + lex // 2


def dag(a):
    return a.mH


def mm(a, b):
    """products of 3x3 matrices, one site at a time (no batched library product)"""
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(3))


def project_su3(u):
    """Gram-Schmidt of the first two columns, the third their cross product"""
    a = u[..., :, 0]
    a = a / torch.linalg.vector_norm(a, dim=-1, keepdim=True)
    b = u[..., :, 1]
    b = b - (a.conj() * b).sum(-1, keepdim=True) * a
    b = b / torch.linalg.vector_norm(b, dim=-1, keepdim=True)
    return torch.stack([a, b, torch.linalg.cross(a, b, dim=-1).conj()], dim=-1)


def make_links(g, gen, sweeps=5, alpha=0.36):
    """list of four (2 volh, 3, 3) link fields"""
    U = [project_su3(torch.randn((2 * g.volh, 3, 3), dtype=torch.complex128, device=DEV, generator=gen))
         for _ in range(4)]
    for _ in range(sweeps):
        new = []
        for mu in range(4):
            s = torch.zeros_like(U[mu])
            for nu in range(4):
                if nu == mu:
                    continue
                f, n, b = g.fwd[mu], g.fwd[nu], g.bwd[nu]
                s += mm(mm(U[nu], U[mu][n]), dag(U[nu][f]))
                s += mm(mm(dag(U[nu][b]), U[mu][b]), U[nu][b][f])
            new.append(project_su3((1 - alpha) * U[mu] + alpha / 6 * s))
        U = new
    return U


def links_to_host(U, volh):
    """the library's host layout (4, 2, volh, column, row, re/im)"""
    u = torch.stack([m.reshape(2, volh, 3, 3).transpose(-1, -2) for m in U])
    return torch.view_as_real(u.contiguous()).cpu().numpy()


def spinor(volh, gen):
    """Gaussian spinor (12, volh, 2), component 3*spin + colour"""
    return torch.randn((12, volh, 2), dtype=torch.float64, device=DEV, generator=gen)


def momenta(volh, gen):
    return torch.randn((4, 2, 8, volh), dtype=torch.float64, device=DEV, generator=gen)


def inputs(case, seed):
    """everything a case is made of, from the seed alone"""
    g = Grid(extents(case))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000003 * (int(seed) % (1 << 40)) + 17)
    d = {"U": make_links(g, gen)}
    vh, kind = g.volh, case["kind"]
    if kind in ("dslash", "apply", "cg", "mixed"):
        d["b"] = spinor(vh, gen)
    elif kind == "multi":
        d["b"] = [spinor(vh, gen) for _ in range(case["nrhs"])]
    elif kind in ("dsf", "md"):
        d["a"] = spinor(vh, gen)
        d["b"] = spinor(vh, gen)
        d["p"] = momenta(vh, gen)
    elif kind == "hmc":
        d["p"] = momenta(vh, gen)
        d["eta1"], d["eta2"] = spinor(vh, gen) * 0.5 ** 0.5, spinor(vh, gen) * 0.5 ** 0.5
    d["f"] = momenta(vh, gen)
    return g, d


def rest_of(b, rel):
    return rel * rel * float((b * b).sum())


# relative residual of the solves: with it the solution, a double, is good to
# nine digits also for the light quark
SOLVE_REL = 1e-12


def mass_list(case):
    """kappa per right-hand side: the masses in turn, the lightest first (0.133, 0.13, 0.12 for three)"""
    k = [case["kappa"], 0.13 if case["kappa"] > 0.13 else 0.118, 0.12][:case["masses"]]
    n = case["nrhs"]
    return [k[j * len(k) // n] for j in range(n)]


def prepare(case, seed):
    L = extents(case)
    g, d = inputs(case, seed)
    lat = bqcd_hip.Lattice(L)
    lat.load_gauge(links_to_host(d.pop("U"), g.volh))
    kappa = case.get("kappa", 0.0)
    if kappa and case["kind"] not in ("multi", "hmc"):
        lat.build_clover(CSW * kappa)
    s = {"case": case, "lat": lat, **d}
    kind = case["kind"]
    if kind in ("dslash", "apply"):
        s["out"] = torch.empty_like(s["b"])
    elif kind in ("cg", "mixed"):
        s["x"] = torch.empty_like(s["b"])
        s["rest"] = rest_of(s["b"], SOLVE_REL)
    elif kind == "multi":
        s["x"] = [torch.empty_like(b) for b in s["b"]]
        s["rests"] = [rest_of(b, SOLVE_REL) for b in s["b"]]
        s["kappas"] = mass_list(case)
    elif kind in ("md", "hmc"):
        lat.gauge_backup(0)
        if kind == "md":
            s["out"] = torch.empty_like(s["a"])
        else:
            s["prm"] = bqcd_hip.hmc_params(
                BETA, kappa, CSW, RHO, 0.05, 2, m_scale=2, model="C", integrator="omelyan",
                rest=1e-24 * 12 * g.volh, maxiter=20000, precision=case["precision"], mre_vectors=4)
    torch.cuda.synchronize()
    return s


def run(s):
    case, lat = s["case"], s["lat"]
    kind = case["kind"]
    if kind == "dslash":
        lat.dslash_d(case["parity"], case["dagger"], s["out"], s["b"])
        return s["out"]
    if kind == "apply":
        lat.apply_d(case["op"], case["kappa"], RHO, s["out"], s["b"])
        return s["out"]
    if kind == "cg":
        s["x"].zero_()
        lat.cg_d(case["op"], s["x"], s["b"], case["kappa"], RHO, rest=s["rest"], maxiter=20000)
        return s["x"]
    if kind == "mixed":
        s["x"].zero_()
        lat.cg_mixed_d(case["op"], s["x"], s["b"], case["kappa"], RHO, rest=s["rest"], maxiter=40000,
                       precision=case["precision"])
        return s["x"]
    if kind == "multi":
        for x in s["x"]:
            x.zero_()
        lat.cg_multi_d("mtdagmt", s["x"], s["b"], s["kappas"], csw=CSW, rests=s["rests"], maxiter=40000,
                       precision=case["precision"])
        return s["x"]
    if kind == "dsf":
        lat.dsf_d(s["f"], s["a"], s["b"], STEP, case["kappa"], CSW * case["kappa"])
        return s["f"]
    if kind == "dsg":
        lat.dsg_d(s["f"], STEP, BETA)
        return s["f"]
    if kind == "md":
        ck = CSW * case["kappa"]
        lat.gauge_restore(0)
        lat.hmc_u_d(s["p"], STEP, ck)
        lat.apply_d("w_mult", case["kappa"], RHO, s["out"], s["a"])
        lat.dsf_d(s["f"], s["a"], s["out"], STEP, case["kappa"], ck)
        lat.dsd_d(s["f"], STEP, ck)
        lat.dsg_d(s["f"], STEP, BETA)
        return [s["f"], s["out"]]
    lat.gauge_restore(0)
    o = lat.hmc_trajectory_d(s["prm"], s["p"], s["eta1"], s["eta2"])
    return {"terms": [o[k] for k in ("h_old", "h_new", "sg_new", "sp_new", "sd_new", "sf1_new", "sf2_new", "plaquette")],
            "links": lat.save_gauge()}


# ---------------------------------------------------------------------------
# the bytes and operations of one pass: every field read or written once
# ---------------------------------------------------------------------------
def work(case):
    vh, kind = sites_per_parity(case), case["kind"]
    links, spin, clov, mom = 8 * 144, 192, 576, 8 * 64  # bytes per site of one parity (links: both parities)
    mt_flops = 2 * HOP_FLOPS + 2 * CLOVER_FLOPS + 48
    if kind == "dslash":
        return {"bytes": vh * (links + 2 * spin), "flops": vh * HOP_FLOPS}
    if kind == "apply":
        n = 2 if case["op"] in ("mtdagmt", "w_dagger_w") else 1
        return {"bytes": vh * (links + 2 * clov + 2 * spin), "flops": vh * n * mt_flops}
    it = vh * (2 * mt_flops + 4 * 48 + 24 * 4)  # one CG iteration

    def iters(kappa):  # to the tolerance, roughly: they grow towards the critical kappa
        return 120 if kappa <= 0.122 else 350 if kappa <= 0.131 else 650

    if kind == "cg":
        return {"bytes": vh * (links + 2 * clov + 3 * spin), "flops": it * iters(case["kappa"])}
    if kind == "mixed":
        return {"bytes": vh * (links + 2 * clov + 3 * spin), "flops": it * iters(case["kappa"])}
    if kind == "multi":
        n = case["nrhs"]
        return {"bytes": vh * (links + 3 * n * spin), "flops": it * sum(iters(k) for k in mass_list(case))}
    m3 = 198  # operations of a 3x3 complex product
    gforce = 8 * (3 * 4 + 1) * m3
    cforce = 8 * 3 * 12 * m3
    if kind == "dsg":
        return {"bytes": vh * (links + 2 * mom), "flops": vh * gforce}
    dsf = 8 * 2 * (2 * m3) + 2 * cforce // 2 + 2 * HOP_FLOPS + 2 * CLOVER_FLOPS
    if kind == "dsf":
        return {"bytes": vh * (links + clov + 2 * spin + 2 * mom), "flops": vh * dsf}
    build = 2 * 6 * 12 * m3 + 2 * 2 * 900
    md = dsf + gforce + cforce + build + 8 * 20 * m3 + mt_flops
    if kind == "md":
        return {"bytes": vh * (2 * links + mom + 2 * spin + 2 * mom), "flops": vh * md}
    # a short trajectory: 17 inner and 5 outer force evaluations, 24 solves
    return {"bytes": vh * (2 * links + mom + 2 * spin), "flops": vh * 17 * md + 24 * it * iters(case["kappa"])}


# ---------------------------------------------------------------------------
# the same results in plain torch, FP64
# ---------------------------------------------------------------------------
def gammas():
    z = torch.zeros((2, 2), dtype=torch.complex128)
    G = [[[0, 1j], [1j, 0]], [[0, 1], [-1, 0]], [[1j, 0], [0, -1j]]]
    out = []
    for m in G:
        m = torch.tensor(m, dtype=torch.complex128)
        out.append(torch.cat([torch.cat([z, m], 1), torch.cat([m.mH, z], 1)], 0).to(DEV))
    out.append(torch.diag(torch.tensor([1, 1, -1, -1], dtype=torch.complex128)).to(DEV))
    return out


def gellmann():
    lam = np.zeros((8, 3, 3), complex)
    lam[0][0, 1] = lam[0][1, 0] = 1
    lam[1][0, 1], lam[1][1, 0] = -1j, 1j
    lam[2][0, 0], lam[2][1, 1] = 1, -1
    lam[3][0, 2] = lam[3][2, 0] = 1
    lam[4][0, 2], lam[4][2, 0] = -1j, 1j
    lam[5][1, 2] = lam[5][2, 1] = 1
    lam[6][1, 2], lam[6][2, 1] = -1j, 1j
    lam[7] = np.diag([1, 1, -2]) / np.sqrt(3)
    return torch.tensor(lam, device=DEV)


def to_sites(v):
    """(12, volh, 2) -> complex (volh, 4, 3)"""
    return torch.view_as_complex(v.contiguous()).reshape(4, 3, -1).permute(2, 0, 1)


def from_sites(v):
    return torch.view_as_real(v.permute(1, 2, 0).reshape(12, -1).contiguous())


def algebra(w):
    """(..., 8, volh) coordinates -> Hermitian (..., volh, 3, 3)"""
    lam = gellmann()
    return sum(w[..., j, :, None, None] * lam[j] for j in range(8))


class Exact:
    """Operators and actions of a link field; differentiable in the links."""

    def __init__(self, g, U):
        self.g, self.U, self.gam = g, U, gammas()

    def hop(self, e, psi, dagger=False):
        """out on parity e from psi on parity 1 - e"""
        g, vh = self.g, self.g.volh
        me = slice(e * vh, (e + 1) * vh)
        sg = 1.0 if dagger else -1.0
        out = 0
        one = torch.eye(4, dtype=torch.complex128, device=DEV)
        for mu in range(4):
            for fwd in (True, False):
                j = (g.fwd if fwd else g.bwd)[mu][me] - (1 - e) * vh
                sign = (g.fsign if fwd else g.bsign)[mu][me]
                P = one + (sg if fwd else -sg) * self.gam[mu]
                h = psi[j] * sign[:, None, None]
                h = sum(P[:, s, None] * h[:, None, s, :] for s in range(4))
                u = self.U[mu][me] if fwd else dag(self.U[mu][(1 - e) * vh:(2 - e) * vh][j])
                out = out + sum(u[:, None, :, c] * h[:, :, c, None] for c in range(3))
        return out

    def field_strength(self, mu, nu):
        g, Um, Un = self.g, self.U[mu], self.U[nu]
        fm, fn, bm, bn = g.fwd[mu], g.fwd[nu], g.bwd[mu], g.bwd[nu]
        q = mm(mm(Um, Un[fm]), dag(mm(Un, Um[fn])))
        q = q + mm(mm(Un, dag(Um[bm][fn])), mm(dag(Un[bm]), Um[bm]))
        q = q + mm(dag(mm(Un[bm][bn], Um[bm])), mm(Um[bm][bn], Un[bn]))
        q = q + mm(mm(dag(Un[bn]), Um[bn]), mm(Un[bn][fm], dag(Um)))
        return (q - dag(q)) / 8j

    def clover(self, csw_kappa):
        """A = 1 - csw kappa sum sigma F as its blocks on psi_up +- psi_low: two (2 volh, 6, 6)"""
        n = 2 * self.g.volh
        P = torch.eye(6, dtype=torch.complex128, device=DEV).expand(n, 6, 6)
        Q = torch.zeros((n, 6, 6), dtype=torch.complex128, device=DEV)
        for mu in range(4):
            for nu in range(mu + 1, 4):
                s = 0.5j * (self.gam[mu] @ self.gam[nu] - self.gam[nu] @ self.gam[mu])
                F = self.field_strength(mu, nu)
                P = P - csw_kappa * (s[:2, None, :2, None] * F[:, None, :, None, :]).reshape(n, 6, 6)
                Q = Q - csw_kappa * (s[:2, None, 2:, None] * F[:, None, :, None, :]).reshape(n, 6, 6)
        return [P + Q, P - Q]

    def set_clover(self, csw_kappa):
        self.A = self.clover(csw_kappa)
        self.I = [inverse6(a)[0] for a in self.A]

    def mult(self, blocks, e, psi):
        vh = self.g.volh
        y = []
        for b, sg in zip(blocks, (1, -1)):
            x = (psi[:, :2] + sg * psi[:, 2:]).reshape(vh, 6) / 2
            a = b[e * vh:(e + 1) * vh]
            y.append(sum(a[:, :, k] * x[:, k, None] for k in range(6)).reshape(vh, 2, 3))
        return torch.cat([y[0] + y[1], y[0] - y[1]], 1)

    def mtil(self, psi, kappa, rho=0.0, dagger=False):
        t = self.mult(self.I, 1, self.hop(1, psi, dagger))
        return self.mult(self.A, 0, psi) - kappa ** 2 * self.hop(0, t, dagger) + rho * psi

    def apply(self, op, psi, kappa, rho):
        r = rho if op.startswith("w_") else 0.0
        if op in ("mtil", "w_mult"):
            return self.mtil(psi, kappa, r)
        if op in ("mtil_dag", "w_mult_dag"):
            return self.mtil(psi, kappa, r, True)
        return self.mtil(self.mtil(psi, kappa, r), kappa, r, True)

    def cg(self, op, b, kappa, rho, rest, maxiter):
        x = torch.zeros_like(b)
        r, p = b.clone(), b.clone()
        rr = float((r.conj() * r).real.sum())
        for _ in range(maxiter):
            q = self.apply(op, p, kappa, rho)
            al = rr / float((p.conj() * q).real.sum())
            x += al * p
            r -= al * q
            new = float((r.conj() * r).real.sum())
            if new <= rest:
                break
            p = r + (new / rr) * p
            rr = new
        return x

    def plaquettes(self):
        g, s = self.g, 0.0
        for mu in range(4):
            for nu in range(mu + 1, 4):
                a = mm(self.U[mu], self.U[nu][g.fwd[mu]])
                b = mm(self.U[nu], self.U[mu][g.fwd[nu]])
                s = s + (a * b.conj()).real.sum()  # Re Tr a b^+
        return s


def inverse6(a):
    """inverse and pivots of Hermitian positive 6x6 matrices (Gauss-Jordan, no pivoting)"""
    n = a.shape[0]
    m = torch.cat([a, torch.eye(6, dtype=a.dtype, device=a.device).expand(n, 6, 6)], 2)
    piv = []
    for k in range(6):
        d = m[:, k, k]
        piv.append(d.real)
        row = m[:, k] / d[:, None]
        rows = [row if r == k else m[:, r] - m[:, r, k, None] * row for r in range(6)]
        m = torch.stack(rows, 1)
    return m[:, :, 6:], piv


def displaced(U, w, volh):
    """U + i (w.lambda) U: first order in w, enough for the derivative at w = 0"""
    return [U[mu] + mm(1j * algebra(w[mu]).reshape(2 * volh, 3, 3), U[mu]) for mu in range(4)]


def force(g, U, action):
    """d action / d w at w = 0"""
    w = torch.zeros((4, 2, 8, g.volh), dtype=torch.float64, device=DEV, requires_grad=True)
    action(Exact(g, displaced(U, w, g.volh))).backward()
    return w.grad


def gauge_force(g, U):
    return force(g, U, lambda E: STEP * BETA / 3.0 * E.plaquettes())


def fermion_force(g, U, a, b, kappa):
    a, b = to_sites(a), to_sites(b)

    def act(E):
        E.set_clover(CSW * kappa)
        return 2.0 * STEP * (b.conj() * E.mtil(a, kappa)).real.sum()
    return force(g, U, act)


def det_force(g, U, kappa):
    vh = g.volh

    def act(E):
        s = 0.0
        for a in E.clover(CSW * kappa):
            s = s + sum(torch.log(d).sum() for d in inverse6(a[vh:])[1])
        return 2.0 * STEP * s
    return force(g, U, act)


def exact(case, seed):
    kind, vh = case["kind"], sites_per_parity(case)
    if kind == "hmc" or (kind in ("cg", "mixed", "multi") and vh > 70000) \
            or (kind == "multi" and vh * case["nrhs"] > 300000):
        return None
    g, d = inputs(case, seed)
    U, kappa = d["U"], case.get("kappa", 0.0)
    if kind == "dsg":
        return d["f"] + gauge_force(g, U)
    if kind == "dsf":
        return d["f"] + fermion_force(g, U, d["a"], d["b"], kappa)
    with torch.no_grad():
        E = Exact(g, U)
        if kind == "dslash":
            return from_sites(E.hop(case["parity"], to_sites(d["b"]), case["dagger"]))
        if kind in ("apply", "cg", "mixed"):
            E.set_clover(CSW * kappa)
            b = to_sites(d["b"])
            if kind == "apply":
                return from_sites(E.apply(case["op"], b, kappa, RHO))
            return from_sites(E.cg(case["op"], b, kappa, RHO, rest_of(d["b"], 1e-13), 5000))
        if kind == "multi":
            xs, last = [], None
            for k, b in zip(mass_list(case), d["b"]):
                if k != last:
                    E.set_clover(CSW * k)
                    last = k
                xs.append(from_sites(E.cg("mtdagmt", to_sites(b), k, 0.0, rest_of(b, 1e-13), 5000)))
            return xs
        # one molecular-dynamics step
        H = algebra(STEP * d["p"]).reshape(4, 2 * vh, 3, 3)
        for mu in range(4):
            t = u = U[mu]
            for n in range(1, 24):
                t = mm(1j * H[mu], t) / n
                u = u + t
            U[mu] = u
        E = Exact(g, U)
        E.set_clover(CSW * kappa)
        out = from_sites(E.mtil(to_sites(d["a"]), kappa, RHO))
    f = d["f"] + fermion_force(g, U, d["a"], out, kappa)
    f = f + det_force(g, U, kappa)
    return [f + gauge_force(g, U), out]
