"""Benchmark: CG time to |r|/|b| <= 1e-10 on one MI355X, and FP64 hopping-matrix
HBM bandwidth.

Workload (the precision configuration): 32^3 x 64 lattice, Haar-random SU(3)
links smoothed by 5 APE-like sweeps (alpha = 0.36 in the (1-alpha) U + alpha/6 sum
of staples convention: plaquette ~0.55), kappa = 0.1355, csw = 1.9,
one unit complex Gaussian source on the even sites, antiperiodic in time.
A step is one solve of M~^+ M~ x = phi from x = 0 to |r|^2 <= 1e-20 |phi|^2
(the reference's absolute float32 bound, cg.F90:111) with every field resident
in HBM.  The solver is selectable; its FP64 true residual is always checked.

Also measured: the FP64 hopping matrix (d, d/D21.F90) in isolation, timed with
HIP events on the stream it is launched on; algorithmic traffic 1536 B/site
(8 links x 144 B + in 192 B + out 192 B).

CPU baseline: the reference BQCD Fortran CG (oracle/_ref, built from the
reference sources with OpenMP) on the same field, a bounded number of
iterations, scaled to the GPU solve's iteration count; when that binary is
absent, the oracle's C restatement is timed instead.
"""
import argparse
import json
import os
import subprocess
import sys
import tempfile
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "bqcd-r399-quda_amd"))

DSLASH_BYTES_PER_SITE = 8 * 144 + 192 + 192
# one FP64 CG iteration on M~^+M~ (cg.F90:93-117) per even site: four fused
# operator kernels (A^-1 D twice: 2112 B each; A x - k^2 D t: 2304 B; the same
# with the dot product against p: 2496 B) and the vector updates (r with |r|^2:
# reads q, r, writes r, 576 B; x and p: reads r, p, x, writes p, x, 960 B);
# with two-row links each operator kernel reads 8 x 96 B of links instead of
# 8 x 144 B
CG_ITER_BYTES_PER_SITE_18 = 2 * 2112 + 2304 + 2496 + 576 + 960
CG_ITER_BYTES_PER_SITE_12 = CG_ITER_BYTES_PER_SITE_18 - 4 * 8 * 48
# 16-bit hopping kernel with the A^-1 epilogue (first half of the mixed solver's
# operator): 8 two-row links of 24 B, the input and output spinors (48 B + 4 B
# norm each), two clover blocks of 18 words (72 B) plus their (m, c) float2
DSLASH16_CLINV_BYTES_PER_SITE = 8 * 24 + 2 * (48 + 4) + 2 * (72 + 8)
# the usual hopping-term count per output site: 8 spin projections, 8 SU(3) x
# half-spinor products, reconstruction and the sum over directions
DSLASH_FLOPS_PER_SITE = 1320
HBM_PEAK_GBS = 8000.0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--lattice", default="32,32,32,64")
    ap.add_argument("--kappa", type=float, default=0.1355)
    ap.add_argument("--csw", type=float, default=1.9)
    ap.add_argument("--solver", default="mixed16", choices=["f64", "mixed32", "mixed16"])
    ap.add_argument("--delta", type=float, default=0.1)
    ap.add_argument("--max-inner", type=int, default=1000)
    ap.add_argument("--dslash-reps", type=int, default=50)
    ap.add_argument("--cpu-iters", type=int, default=200,
                    help="reference CG iterations timed on the host cores for each CPU baseline")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-sweep", action="store_true",
                    help="skip the precision comparison at the configuration's reliable-update "
                         "settings (FP32 and 16-bit inner, update every 100 iterations or on a "
                         "1e-2 residual drop)")
    ap.add_argument("--no-batch", action="store_true",
                    help="skip the multi-RHS workload (24^3x48, 12 RHS over 3 kappa)")
    ap.add_argument("--batch-lattice", default="24,24,24,48")
    ap.add_argument("--seed", type=int, default=20261202)
    ap.add_argument("--sweeps", type=int, default=5)
    ap.add_argument("--alpha", type=float, default=0.36)
    ap.add_argument("--only-mixed", type=int, default=0, metavar="MAXITER",
                    help="run only one mixed-precision solve (--solver) stopped after MAXITER inner "
                         "iterations (for hardware-counter runs), then exit")
    ap.add_argument("--only-dslash", type=int, default=0,
                    help="run only N FP64 hopping-matrix launches and a calibration copy of the "
                         "same byte count (for hardware-counter runs), then exit")
    ap.add_argument("--only-batch", action="store_true",
                    help="run only the multi-RHS workload (24^3x48, 12 RHS over 3 kappa), print its "
                         "report, then exit (for hardware-counter runs)")
    ap.add_argument("--hmc", type=int, default=0, metavar="NTRAJ",
                    help="run NTRAJ HMC trajectories of the trajectory workload (two Hasenbusch "
                         "pseudofermions, Omelyan, tau=1, 20 outer steps, from a start thermalised "
                         "on --hmc-tile) with the solvers of --hmc-runs (16-bit mixed precision and "
                         "FP64 by default), print the report, then exit")
    ap.add_argument("--hmc-lattice", default="48,48,48,96")
    ap.add_argument("--hmc-kappa", type=float, default=0.1365)
    ap.add_argument("--hmc-rho", type=float, default=0.1)
    ap.add_argument("--hmc-steps", default="20",
                    help="outer steps per trajectory; a comma list runs the trajectories once per "
                         "step count from the same start (the step-size scaling of Delta H)")
    ap.add_argument("--hmc-mscale", type=int, default=2, help="inner steps per outer step")
    ap.add_argument("--hmc-model", default="C", choices=["B", "C"],
                    help="Hasenbusch time-scale split (hmc_integrator.F90): B = both pseudofermion "
                         "forces on the outer steps; C = the rho-shifted one with the gauge force on "
                         "the inner steps")
    ap.add_argument("--hmc-therm", type=int, default=60,
                    help="force-accepted trajectories of length 0.5 from the smeared start (on the "
                         "--hmc-tile lattice when given) before the measured ones")
    ap.add_argument("--hmc-tile", default="16,16,16,32", metavar="LATTICE",
                    help="make the start on this smaller lattice (smearing, --hmc-quench, "
                         "--hmc-therm) and repeat its links periodically to fill --hmc-lattice "
                         "(each of its extents must divide the full one); empty: start on the "
                         "full lattice")
    ap.add_argument("--hmc-quench", type=int, default=0, metavar="NTRAJ",
                    help="pure-gauge molecular-dynamics trajectories (tau 1, 20 steps, fresh momenta "
                         "each, no accept/reject) at --hmc-quench-beta before the dynamical "
                         "thermalisation: they give the smeared start equilibrium-like short-distance "
                         "fluctuations at the cost of gauge forces only")
    ap.add_argument("--hmc-quench-beta", type=float, default=5.7)
    ap.add_argument("--hmc-therm-steps", type=int, default=10,
                    help="outer steps of each thermalisation trajectory")
    ap.add_argument("--hmc-mre", type=int, default=4,
                    help="chronological initial-guess vectors per pseudofermion (mre.F90)")
    ap.add_argument("--hmc-first", type=int, default=0,
                    help="index of the first measured trajectory (its draws and accept number): "
                         "a run split over several jobs continues where the last one stopped")
    ap.add_argument("--hmc-restart", action="store_true",
                    help="start every measured trajectory from the thermalised start (independent "
                         "proposals with their own draws) instead of chaining them; a run split over "
                         "several jobs (--hmc-first) then gives the same trajectories as one job")
    ap.add_argument("--hmc-runs", default="mixed16,fp64",
                    help="solver runs of the trajectory workload, comma separated "
                         "(mixed16, mixed32, fp64, and mixed16_batched / mixed32_batched, which solve "
                         "the two pseudofermion systems together where they meet at the same links: "
                         "slower, since the shifted system converges first and its lanes stay masked "
                         "in the block)")
    ap.add_argument("--reference-workload", choices=["smp", "mpp"], default=None,
                    help="run the reference's own benchmark input (work/input.smp: 24^3x48, one "
                         "trajectory of 10 leapfrog steps; work/input.mpp: 48^3x96, two trajectories "
                         "of 20 steps; beta 5, kappa 0.13, csw 1.923, cold start, every CG stopped "
                         "after 100 iterations) on the GPU, and for smp the reference hmc() on the "
                         "host cores (unless --no-cpu); print the timings, then exit")
    ap.add_argument("--scan", action="store_true",
                    help="print plaquette and FP64 iteration counts per smearing sweep, then exit")
    return ap.parse_args()


def measured_traffic(L, kind="fp64"):
    """HBM bytes per launch of the FP64 hopping matrix (kind "fp64") or the
    16-bit A^-1 D kernel ("f16") from the committed rocprofv3 FETCH_SIZE /
    WRITE_SIZE summary (calibrated against a device copy), for the lattice
    that summary covers; None otherwise."""
    path = os.path.join(REPO, "profiles", "dslash_%s_%s.md" % (kind, "x".join(map(str, L))))
    if not os.path.exists(path):
        return None, None
    for line in open(path):
        if line.startswith("traffic_bytes_per_launch:"):
            return float(line.split(":")[1]), os.path.relpath(path, REPO)
    return None, None


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def tile_links(us, Ls, L):
    """Links of the lattice L (host layout [mu][eo][site][3][3][2], BQCD's
    even-odd site index i = (x + Lx (y + Ly (z + Lz t))) / 2) built by repeating
    those of the smaller lattice Ls periodically: U_mu(x) = U_small_mu(x mod Ls).
    The extents are even, so a site and its image have the same parity, and
    every plaquette of L is a copy of one of Ls."""
    import numpy as np

    if any(n % s or s % 2 for n, s in zip(L, Ls)):
        raise ValueError("cannot tile %r with %r" % (L, Ls))
    vh = L[0] * L[1] * L[2] * L[3] // 2
    out = np.empty((4, 2, vh) + us.shape[3:], dtype=us.dtype)
    x = np.arange(L[0])[None, None, :]
    y = np.arange(L[1])[None, :, None]
    z = np.arange(L[2])[:, None, None]
    for t in range(L[3]):
        j = (x + L[0] * (y + L[1] * (z + L[2] * t))).ravel()
        eo = ((x + y + z + t) & 1).ravel()
        xs, ys, zs, ts = x % Ls[0], y % Ls[1], z % Ls[2], t % Ls[3]
        js = (xs + Ls[0] * (ys + Ls[1] * (zs + Ls[2] * ts))).ravel()
        out[:, eo, j >> 1] = us[:, eo, js >> 1]
    return out


def cpu_model():
    """the host CPU's model name and the number of logical CPUs this process may use"""
    name = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    name = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return name, len(os.sched_getaffinity(0))


def cpu_threads():
    return int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or len(os.sched_getaffinity(0))


def raise_stack_limit():
    """child set-up for the reference's OpenMP programs: the main thread's stack
    raised to the hard limit (at 24^3x48 with 16 threads the reference's
    trajectory overflows the usual 8 MiB)"""
    import resource

    soft, hard = resource.getrlimit(resource.RLIMIT_STACK)
    resource.setrlimit(resource.RLIMIT_STACK, (hard, hard))


def cpu_baseline(g, b_dev, kappa, csw, gpu_iters, cpu_iters, what="the GPU FP64 solve"):
    """Times the reference Fortran CG (or the oracle) on the same field: cpu_iters
    iterations, scaled to gpu_iters."""
    import numpy as np

    ref = os.path.join(REPO, "oracle", "_ref", "bqcd_golden_omp")
    threads = cpu_threads()
    model, ncpu = cpu_model()
    L = g.L
    lat_s = "x".join(map(str, L))
    if os.path.exists(ref):
        with tempfile.TemporaryDirectory(dir="/tmp") as d:
            u = g.save_gauge(flipped=False)
            u.tofile(os.path.join(d, "u.bin"))
            del u
            eta = g.to_host(b_dev)
            eta.tofile(os.path.join(d, "eta_e.bin"))
            np.zeros_like(eta).tofile(os.path.join(d, "eta_o.bin"))
            ctl = "%d %d %d %d\n%.17g %.17g 0\n1e-30 %d\n0 0\n%s\n%s\n%d\n" % (
                *L, kappa, csw, cpu_iters, d, d, cpu_iters)
            env = dict(os.environ, OMP_NUM_THREADS=str(threads))
            t0 = time.time()
            p = subprocess.run([ref], input=ctl.encode(), capture_output=True, env=env, timeout=900,
                               preexec_fn=raise_stack_limit)
            wall = time.time() - t0
            out = p.stdout.decode()
            if p.returncode != 0:
                raise RuntimeError("reference CPU run failed: %s %s" % (out, p.stderr.decode()))
            tok = out.split()
            cg_s = float(tok[tok.index("cg_seconds") + 1])
            it = int(tok[tok.index("cg_iters") + 1])
        per_iter = cg_s / it
        return {
            "value": per_iter * gpu_iters,
            "unit": "s",
            "cores": threads,
            "kind": "reference",
            "cpu_model": model,
            "cpus_available": ncpu,
            "ms_per_iteration": 1e3 * per_iter,
            "sample": "reference BQCD Fortran cg() (libd21, single_pe, OpenMP, amdflang -O2) "
                      "on the same %s field, %d OpenMP threads on %s: %d iterations in %.2f s "
                      "(%.1f ms/iter, process wall %.1f s incl. clover_init and I/O), scaled to "
                      "the %d iterations of %s" % (lat_s, threads, model, it, cg_s, 1e3 * per_iter,
                                                  wall, gpu_iters, what),
        }
    # oracle port (single thread: a second per iteration at 32^3x64)
    cpu_iters = min(cpu_iters, 20)
    sys.path.insert(0, os.path.join(REPO, "tests"))
    import oracle_lib as ol

    lat = ol.Lattice(L)
    u = g.save_gauge(flipped=False)
    a, ai, bcl = lat.clover_init(u, csw * kappa)
    op = lat.op(lat.flip_bc(u), a, ai, kappa, csw * kappa)
    eta = g.to_host(b_dev)
    t0 = time.time()
    lat.cg(op, 2, eta, 1e-30, cpu_iters)
    dt = time.time() - t0
    return {"value": dt / cpu_iters * gpu_iters, "unit": "s", "cores": 1, "kind": "port",
            "cpu_model": model, "cpus_available": ncpu, "ms_per_iteration": 1e3 * dt / cpu_iters,
            "sample": "oracle C restatement cg() on the same %s field, 1 thread on %s: %d iterations "
                      "in %.2f s, scaled to the %d iterations of %s"
                      % (lat_s, model, cpu_iters, dt, gpu_iters, what)}


def batched(args, torch, dev, stream):
    """Multi-RHS workload: 12 right-hand sides over 3 Hasenbusch kappa values
    (0.1355, 0.13, 0.12; 4 Gaussian sources each), csw 1.9, tolerance
    |r|/|b| <= 1e-10 each; the block solver (autotuned RHS block) against 12
    sequential single-RHS solves with the same mixed-precision solver and with
    the FP64 solver."""
    import bqcd_hip

    L = tuple(int(v) for v in args.batch_lattice.split(","))
    kappas = [0.1355] * 4 + [0.13] * 4 + [0.12] * 4
    g = bqcd_hip.Lattice(L)
    g.set_stream(stream)
    g.gauge_random(args.seed + 7, 0.0)
    g.gauge_smear(args.sweeps, args.alpha)
    plaq = g.plaquette()
    gen = torch.Generator(device=dev)
    gen.manual_seed(args.seed + 8)
    bs = [torch.randn((12, g.volh, 2), dtype=torch.float64, device=dev, generator=gen) * (0.5 ** 0.5)
          for _ in kappas]
    xs = [torch.zeros_like(b) for b in bs]
    rests = [1e-20 * float((b * b).sum()) for b in bs]
    prec = "f16" if args.solver != "mixed32" else "f32"

    def timed(fn):
        torch.cuda.synchronize()
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        t0.record(stream)
        out = fn()
        t1.record(stream)
        torch.cuda.synchronize()
        return t0.elapsed_time(t1) / 1e3, out

    def sequential(mixed):
        its = []
        for k, kap in enumerate(kappas):
            if k == 0 or kap != kappas[k - 1]:
                g.build_clover(args.csw * kap)
            xs[k].zero_()
            if mixed:
                it, _, tr = g.cg_mixed_d("mtdagmt", xs[k], bs[k], kap, rest=rests[k], maxiter=40000,
                                         precision=prec, delta=args.delta, max_inner=args.max_inner)
            else:
                it, tr = g.cg_d("mtdagmt", xs[k], bs[k], kap, rest=rests[k], maxiter=40000)
            its.append(it)
        return its

    def block_solve():
        for x in xs:
            x.zero_()
        return g.cg_multi_d("mtdagmt", xs, bs, kappas, csw=args.csw, rests=rests, maxiter=40000,
                            precision=prec, block=0)

    block_solve()  # autotunes the RHS block and workgroup sizes (cached per lattice and precision)
    t_blk, (its_blk, trs_blk, blk) = timed(block_solve)
    tile = g.multi_tile()
    x_blk = [x.clone() for x in xs]
    t_seq_mixed, its_seq = timed(lambda: sequential(True))
    t_seq_f64, its_f64 = timed(lambda: sequential(False))
    err = max(float(torch.linalg.vector_norm(x_blk[k] - xs[k]) / torch.linalg.vector_norm(xs[k]))
              for k in range(len(kappas)))
    res = {
        "lattice": list(L), "plaquette": round(plaq, 6), "nrhs": len(kappas), "kappas": kappas,
        "csw": args.csw, "precision": prec, "block_size": blk, "workgroup_size": tile,
        "block_solve_s": t_blk, "sequential_mixed_s": t_seq_mixed, "sequential_fp64_s": t_seq_f64,
        "speedup_vs_sequential_mixed": t_seq_mixed / t_blk,
        "speedup_vs_sequential_fp64": t_seq_f64 / t_blk,
        "iterations_block": its_blk, "iterations_sequential_fp64": its_f64,
        "max_true_residual_rel": max(trs_blk[k] / (rests[k] * 1e20) for k in range(len(kappas))),
        "max_solution_rel_error_vs_fp64": err,
    }
    if not args.no_cpu:
        # the reference CG's time per iteration on this field (the operator costs
        # the same for every kappa), times the iterations of the 12 FP64 solves
        try:
            res["cpu_baseline"] = cpu_baseline(g, bs[0], kappas[0], args.csw, sum(its_f64), args.cpu_iters,
                                               "the 12 sequential FP64 GPU solves")
        except Exception as exc:  # reported, never silently replaced
            log("batched cpu baseline failed:", exc)
            res["cpu_baseline"] = None
    log("batched:", json.dumps(res))
    g.close()
    return res


def hmc_lattices(args):
    """the trajectory lattice and the lattice its start is made on (None: the same)"""
    L = tuple(int(v) for v in args.hmc_lattice.split(","))
    Ls = tuple(int(v) for v in args.hmc_tile.split(",")) if args.hmc_tile else None
    if Ls and (len(Ls) != 4 or any(n % s or s % 2 for n, s in zip(L, Ls))):
        raise SystemExit("--hmc-tile %s does not divide --hmc-lattice %s into even extents: give "
                         "one that does, or --hmc-tile '' to start on the full lattice"
                         % (args.hmc_tile, args.hmc_lattice))
    return L, Ls


def hmc(args, torch, dev, stream):
    """HMC trajectories: Wilson gauge action beta 5.29, clover csw 1.9, two
    Hasenbusch pseudofermions (S_f1 with W = M~ + rho, S_f2 the ratio),
    Omelyan integrator, trajectory length 1 in --hmc-steps outer steps with
    --hmc-mscale inner steps each (model B: the gauge force inside, both
    pseudofermion forces outside; model C: S_f1 and the clover determinant
    move inside), Gaussian momenta and noise from the device generator,
    Metropolis accept/reject.  The same trajectories (same start, same draws)
    run with each solver of --hmc-runs."""
    import bqcd_hip

    L, Ls = hmc_lattices(args)
    beta, kappa, csw, rho = 5.29, args.hmc_kappa, args.csw, args.hmc_rho
    rng = __import__("random").Random(args.seed + 12)

    def draws(lat):
        return (torch.empty((4, 2, 8, lat.volh), dtype=torch.float64, device=dev),
                torch.empty((12, lat.volh, 2), dtype=torch.float64, device=dev),
                torch.empty((12, lat.volh, 2), dtype=torch.float64, device=dev))

    def make_start(lat):
        """smeared Haar links, pure-gauge trajectories, force-accepted dynamical ones"""
        lat.gauge_random(args.seed + 11, 0.0)
        lat.gauge_smear(args.sweeps, args.alpha)
        p, eta1, eta2 = draws(lat)
        log("hmc start (%s): plaquette %.6f after %d smearing sweeps"
            % ("x".join(map(str, lat.L)), lat.plaquette(), args.sweeps))
        t0 = time.perf_counter()
        dt, nstep = 0.05, 20
        for k in range(args.hmc_quench):
            # leapfrog of hmc_leap_frog.F90 with the gauge force only
            lat.gaussian_d(p, args.seed + 5000 + k, 1.0)
            lat.dsg_d(p, 0.5 * dt, args.hmc_quench_beta)
            for s in range(nstep):
                lat.hmc_u_d(p, dt, 0.0)
                lat.dsg_d(p, dt if s < nstep - 1 else 0.5 * dt, args.hmc_quench_beta)
            if k % 5 == 4 or k == args.hmc_quench - 1:
                torch.cuda.synchronize()
                log("hmc pure-gauge trajectory %d (beta %.3f): plaquette %.6f, %.1f s"
                    % (k, args.hmc_quench_beta, lat.plaquette(), time.perf_counter() - t0))
        # the smeared start is far from equilibrium at beta 5.29: force-accepted
        # trajectories (as the reference's hmc_accept_first) bring it closer
        therm = bqcd_hip.hmc_params(beta=beta, kappa=kappa, csw=csw, rho=rho, tau=0.5 / args.hmc_therm_steps,
                                    ntau=args.hmc_therm_steps, m_scale=args.hmc_mscale, model=args.hmc_model,
                                    integrator="omelyan", rest=1e-20 * 12 * lat.volh, maxiter=50000,
                                    precision="f16", mre_vectors=args.hmc_mre, batch=False, verbose=True)
        for k in range(args.hmc_therm):
            seed = args.seed + 7000 + 100 * k
            lat.gaussian_d(p, seed + 1, 1.0)
            lat.gaussian_d(eta1, seed + 2, 0.5)
            lat.gaussian_d(eta2, seed + 3, 0.5)
            out = lat.hmc_trajectory_d(therm, p, eta1, eta2, accept_random=-1.0)
            log("hmc thermalisation %d: dH %.4f plaquette %.6f, %.1f s"
                % (k, out["h_new"] - out["h_old"], out["plaquette"], out["seconds"]))
        del p, eta1, eta2

    g = bqcd_hip.Lattice(L)
    g.set_stream(stream)
    vh = g.volh
    if Ls:
        gs = bqcd_hip.Lattice(Ls)
        gs.set_stream(stream)
        make_start(gs)
        g.load_gauge(tile_links(gs.save_gauge(), Ls, L))
        gs.close()
        log("hmc start: the links repeated %s times: plaquette %.12f"
            % ("x".join(str(n // s) for n, s in zip(L, Ls)), g.plaquette()))
    else:
        make_start(g)
    p, eta1, eta2 = draws(g)
    rest = 1e-20 * 12 * vh  # |r|/|b| ~ 1e-10 for the unit-variance sources
    g.gauge_backup(1)
    runs = {}
    solvers = {"mixed16_batched": ("f16", True), "mixed32_batched": ("f32", True), "mixed16": ("f16", False),
               "mixed32": ("f32", False), "fp64": ("f64", False)}
    # one accept/reject number per trajectory, shared by every run
    accept_u = [rng.random() for _ in range(args.hmc_first + args.hmc)][args.hmc_first:]
    steps = [int(v) for v in args.hmc_steps.split(",")]
    for nsteps, name in [(n, r) for n in steps for r in args.hmc_runs.split(",")]:
        prec, batch = solvers[name]
        key = name if len(steps) == 1 else "%s@%d" % (name, nsteps)
        g.gauge_restore(1)
        prm = bqcd_hip.hmc_params(beta=beta, kappa=kappa, csw=csw, rho=rho, tau=1.0 / nsteps,
                                  ntau=nsteps, m_scale=args.hmc_mscale, model=args.hmc_model,
                                  integrator="omelyan", rest=rest, maxiter=50000, precision=prec,
                                  mre_vectors=args.hmc_mre, batch=batch, verbose=True)
        trajs = []
        for k in range(args.hmc):
            if args.hmc_restart and k > 0:
                g.gauge_restore(1)
            seed = args.seed + 100 * (args.hmc_first + k)
            g.gaussian_d(p, seed + 1, 1.0)
            g.gaussian_d(eta1, seed + 2, 0.5)
            g.gaussian_d(eta2, seed + 3, 0.5)
            out = g.hmc_trajectory_d(prm, p, eta1, eta2, accept_random=accept_u[k])
            log("hmc %s trajectory %d: dH %.6f exp(-dH) %.6f plaquette %.6f accepted %d, %d CG calls, "
                "%d iterations, %.1f s" % (key, args.hmc_first + k, out["h_new"] - out["h_old"], out["exp_dh"],
                                           out["plaquette"], out["accepted"], out["cg_ncall"],
                                           out["cg_niter_tot"], out["seconds"]))
            log("    dH terms: beta*sg %.4f sp %.4f sd %.4f sf1 %.4f sf2 %.4f"
                % (beta * (out["sg_new"] - out["sg_old"]), out["sp_new"] - out["sp_old"],
                   out["sd_new"] - out["sd_old"], out["sf1_new"] - out["sf1_old"],
                   out["sf2_new"] - out["sf2_old"]))
            trajs.append(out)
        runs[key] = {
            "delta_h": [t["h_new"] - t["h_old"] for t in trajs],
            "plaquette": [t["plaquette"] for t in trajs],
            "acceptance": sum(t["accepted"] for t in trajs) / max(1, len(trajs)),
            "s_per_trajectory": sum(t["seconds"] for t in trajs) / max(1, len(trajs)),
            "cg_iterations_per_trajectory": sum(t["cg_niter_tot"] for t in trajs) / max(1, len(trajs)),
            "force_evaluations_ir_uv": [trajs[0]["n_force_ir"], trajs[0]["n_force_uv"]] if trajs else None,
        }
    res = {"workload": "HMC trajectories, clover-Wilson Nf=2 with two Hasenbusch pseudofermions, %s"
                       % "x".join(map(str, L)),
           "lattice": list(L), "beta": beta, "kappa": kappa, "csw": csw, "rho": rho,
           "integrator": "Omelyan (2MN), tau 1, %s outer steps, %d inner steps each"
                         % (args.hmc_steps, args.hmc_mscale), "mre_vectors": args.hmc_mre,
           "model": args.hmc_model,
           "trajectories": args.hmc, "first_trajectory": args.hmc_first,
           "each_from_start": args.hmc_restart,
           "thermalisation": "%s%s%d force-accepted trajectories of length 0.5 in %d steps%s"
                             % ("on %s: " % args.hmc_tile.replace(",", "x") if args.hmc_tile else "",
                                "%d pure-gauge MD trajectories at beta %.3f, then " % (args.hmc_quench, args.hmc_quench_beta)
                                if args.hmc_quench else "", args.hmc_therm, args.hmc_therm_steps,
                                ", links then repeated periodically" if args.hmc_tile else ""),
           "runs": runs,
           "accept_random": accept_u}
    mixed = next((k for k in ("mixed16", "mixed16_batched") if k in runs), None)
    if "fp64" in runs and mixed:
        res["speedup_vs_fp64"] = runs["fp64"]["s_per_trajectory"] / runs[mixed]["s_per_trajectory"]
    g.close()
    return res


def reference_workload(args, torch, dev, stream):
    """The reference's own benchmark inputs, work/input.smp and work/input.mpp:
    beta 5.0, kappa 0.13, csw 1.923076923076923, model A (no Hasenbusch),
    leapfrog, cold start, solver_rest 1e-99, solver_maxiter 100 and
    solver_ignore_no_convergence 2, so that every CG runs exactly 100
    iterations.  smp: 24^3x48, one force-accepted trajectory of 10 steps of
    0.02 (11 CG calls); mpp: 48^3x96, two trajectories of 20 steps of 0.01
    (21 CG calls each), the first force-accepted.  The FP64 drop-in path runs
    them; momenta and noise come from the device generator (the reference
    draws its own: the work is fixed by the input, the draws move only the end
    point).  Time per trajectory as the library measures it.  For smp the
    reference hmc() itself (oracle/_ref/bqcd_traj_omp, built from the
    reference sources with OpenMP) runs the same input on the host cores."""
    import numpy as np
    import bqcd_hip

    cases = {"smp": ((24, 24, 24, 48), 10, 0.02, 1), "mpp": ((48, 48, 48, 96), 20, 0.01, 2)}
    L, ntau, tau, ntraj = cases[args.reference_workload]
    beta, kappa, csw = 5.0, 0.13, 1.923076923076923
    g = bqcd_hip.Lattice(L)
    g.set_stream(stream)
    vh = g.volh

    def cold():
        u = np.zeros((4, 2, vh, 3, 3, 2))
        for k in range(3):
            u[:, :, :, k, k, 0] = 1.0
        return u

    g.load_gauge(cold())
    prm = bqcd_hip.hmc_params(beta=beta, kappa=kappa, csw=csw, rho=0.0, tau=tau, ntau=ntau, m_scale=1,
                              model="A", integrator="leapfrog", rest=1e-99, maxiter=100, log=2,
                              mre_vectors=0)
    p = torch.empty((4, 2, 8, vh), dtype=torch.float64, device=dev)
    eta = torch.empty((12, vh, 2), dtype=torch.float64, device=dev)
    trajs = []
    for k in range(ntraj):
        g.gaussian_d(p, args.seed + 31 + 10 * k, 1.0)
        g.gaussian_d(eta, args.seed + 32 + 10 * k, 0.5)
        out = g.hmc_trajectory_d(prm, p, eta, accept_random=-1.0 if k == 0 else 0.5)
        log("reference workload %s trajectory %d: %d CG calls, %d iterations (max %d), plaquette %.10f, "
            "%.2f s" % (args.reference_workload, k, out["cg_ncall"], out["cg_niter_tot"], out["cg_niter_max"],
                        out["plaquette"], out["seconds"]))
        trajs.append({"seconds": out["seconds"], "cg_calls": out["cg_ncall"], "cg_iterations": out["cg_niter_tot"],
                      "cg_iterations_max": out["cg_niter_max"], "plaquette": out["plaquette"],
                      "accepted": out["accepted"]})
    del p, eta
    g.close()
    res = {"workload": "work/input.%s of the reference: %s, beta %g, kappa %g, csw %.6f, model A, leapfrog "
                       "%d x %g, cold start, CGs of exactly 100 iterations"
                       % (args.reference_workload, "x".join(map(str, L)), beta, kappa, csw, ntau, tau),
           "gpu": {"path": "FP64 drop-in (hb_hmc_trajectory_d)", "trajectories": trajs,
                   "seconds_total": sum(t["seconds"] for t in trajs)}}
    if args.reference_workload == "smp" and not args.no_cpu:
        ref = os.path.join(REPO, "oracle", "_ref", "bqcd_traj_omp")
        if not os.path.exists(ref):
            res["cpu"] = None
            log("reference workload: %s not built, no CPU run" % ref)
        else:
            threads = cpu_threads()
            model, ncpu = cpu_model()
            with tempfile.TemporaryDirectory(dir="/tmp") as d:
                cold().astype("<f8").tofile(os.path.join(d, "u.bin"))
                ctl = "%d %d %d %d\n%.17g %.17g %.17g 0\n%.17g %d 1 A\n1e-99 100 0 2\n0\n%s\n%s\n" % (
                    *L, beta, kappa, csw, tau, ntau, d, d)
                env = dict(os.environ, OMP_NUM_THREADS=str(threads))
                t0 = time.time()
                r = subprocess.run([ref], input=ctl.encode(), capture_output=True, env=env, cwd=d, timeout=1000,
                                   preexec_fn=raise_stack_limit)
                wall = time.time() - t0
                if r.returncode != 0:
                    raise RuntimeError("reference trajectory failed (exit status %d): %s %s"
                                       % (r.returncode, r.stdout.decode()[-500:], r.stderr.decode()[-500:]))
                info = dict(line.split() for line in open(os.path.join(d, "info.txt")))
            res["cpu"] = {"kind": "reference", "program": "reference hmc() (traj driver, libd21, single_pe, "
                                                          "OpenMP, amdflang -O2), its own draws",
                          "cores": threads, "cpu_model": model, "cpus_available": ncpu,
                          "seconds": wall, "cg_calls": int(float(info["cg_ncall"])),
                          "cg_iterations": int(float(info["cg_niter_tot"])),
                          "note": "process wall time, including reading the 24^3x48 start links"}
            log("reference workload smp on the host: %.1f s, %d threads (%s)" % (wall, threads, model))
    return res


def scan(g, args, torch, dev):
    """plaquette and FP64 CG iterations after each smearing sweep"""
    gen = torch.Generator(device=dev)
    gen.manual_seed(1)
    b = torch.randn((12, g.volh, 2), dtype=torch.float64, device=dev, generator=gen)
    x = torch.zeros_like(b)
    g.gauge_random(args.seed, 0.0)
    for sw in range(0, 9):
        if sw:
            g.gauge_smear(1, args.alpha)
        g.build_clover(args.csw * args.kappa)
        x.zero_()
        it, tr = g.cg_d("mtdagmt", x, b, args.kappa, rest=1e-20 * float((b * b).sum()),
                        maxiter=3000, log=2)
        log("sweeps %d alpha %.2f plaquette %.5f  FP64 CG iters %d  true rel %.2e"
            % (sw, args.alpha, g.plaquette(), it, tr / float((b * b).sum())))
    return 0


def main():
    args = parse()
    if args.gpus != 1:
        print("bench.py measures one GPU: the library runs on a single MI355X "
              "(multi-GPU sharding is designed but not implemented); use --gpus 1",
              file=sys.stderr)
        return 2
    import torch
    import bqcd_hip

    if args.reference_workload:
        dev = torch.device("cuda:0")
        torch.cuda.set_device(dev)
        stream = torch.cuda.Stream(device=dev)
        torch.cuda.set_stream(stream)
        print(json.dumps({"reference_workload": reference_workload(args, torch, dev, stream)}), flush=True)
        return 0

    if args.hmc:
        hmc_lattices(args)  # argument errors before any GPU work
        dev = torch.device("cuda:0")
        torch.cuda.set_device(dev)
        stream = torch.cuda.Stream(device=dev)
        torch.cuda.set_stream(stream)
        print(json.dumps({"hmc": hmc(args, torch, dev, stream)}), flush=True)
        return 0

    if args.only_batch:
        dev = torch.device("cuda:0")
        torch.cuda.set_device(dev)
        stream = torch.cuda.Stream(device=dev)
        torch.cuda.set_stream(stream)
        print(json.dumps({"batched": batched(args, torch, dev, stream)}), flush=True)
        return 0

    L = tuple(int(x) for x in args.lattice.split(","))
    kappa, csw = args.kappa, args.csw
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    # one explicit stream (default priority) for torch and the library, so that
    # torch's events time exactly the library's launches
    stream = torch.cuda.Stream(device=dev)
    torch.cuda.set_stream(stream)

    g = bqcd_hip.Lattice(L, bc=(1, 1, 1, -1), device=0)
    g.set_stream(stream)
    vh = g.volh
    log("lattice", L, "volh", vh)
    g.gauge_random(args.seed, 0.0)
    g.gauge_smear(args.sweeps, args.alpha)
    plaq = g.plaquette()
    if args.scan:
        return scan(g, args, torch, dev)
    g.build_clover(csw * kappa)
    log("plaquette <ReTr U_p>/3 = %.6f" % plaq)

    gen = torch.Generator(device=dev)
    gen.manual_seed(args.seed + 1)
    b = torch.randn((12, vh, 2), dtype=torch.float64, device=dev, generator=gen) * (0.5 ** 0.5)
    x = torch.zeros_like(b)
    bnorm2 = float((b * b).sum())
    rest = 1e-20 * bnorm2

    # ---- FP64 hopping matrix in isolation -----------------------------------
    out = torch.empty_like(b)
    inp = torch.randn((12, vh, 2), dtype=torch.float64, device=dev, generator=gen)
    for _ in range(5):
        g.dslash_d(0, False, out, inp)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(args.dslash_reps):
        g.dslash_d(0, False, out, inp)
    e1.record(stream)
    torch.cuda.synchronize()
    ds_ms = e0.elapsed_time(e1) / args.dslash_reps
    ds_bytes = DSLASH_BYTES_PER_SITE * vh
    ds_gbs = ds_bytes / (ds_ms * 1e-3) / 1e9
    log("FP64 dslash: %.4f ms/launch, %.1f GB/s algorithmic, %.1f GFlop/s"
        % (ds_ms, ds_gbs, DSLASH_FLOPS_PER_SITE * vh / (ds_ms * 1e-3) / 1e9))
    if args.only_dslash:
        for _ in range(args.only_dslash):
            g.dslash_d(0, False, out, inp)
        # calibration: a plain device copy moving exactly ds_bytes (read + write)
        src = torch.empty(ds_bytes // 16, dtype=torch.float64, device=dev)
        dst = torch.empty_like(src)
        for _ in range(args.only_dslash):
            dst.copy_(src)
        torch.cuda.synchronize()
        log("calibration copy: %d bytes read + %d bytes written per launch" % (ds_bytes // 2, ds_bytes // 2))
        # the 16-bit hopping kernel of the mixed solver (A^-1 D), timed the same way
        ms16 = g.time_dslash_lp(b, "f16", reps=args.dslash_reps)
        log("16-bit dslash (A^-1 D): %.4f ms/launch, %.1f GB/s algorithmic"
            % (ms16, DSLASH16_CLINV_BYTES_PER_SITE * vh / (ms16 * 1e-3) / 1e9))
        return 0
    del out, inp

    # ---- solves ---------------------------------------------------------------
    # the FP64 CG iterates with two-row links (row 2 rebuilt; the smeared links
    # are SU(3)); the 18-real form is timed once beside it
    g.set_link_recon(12)

    def solve_f64():
        x.zero_()
        it, tr = g.cg_d("mtdagmt", x, b, kappa, rest=rest, maxiter=20000)
        return it, 0, tr

    def solve_mixed():
        x.zero_()
        return g.cg_mixed_d("mtdagmt", x, b, kappa, rest=rest, maxiter=40000,
                            precision="f16" if args.solver == "mixed16" else "f32",
                            delta=args.delta, max_inner=args.max_inner)

    solve = solve_f64 if args.solver == "f64" else solve_mixed
    if args.only_mixed:
        x.zero_()
        it, nrel, tr = g.cg_mixed_d("mtdagmt", x, b, kappa, rest=rest, maxiter=args.only_mixed, log=2,
                                    precision="f16" if args.solver != "mixed32" else "f32",
                                    delta=args.delta, max_inner=args.max_inner)
        torch.cuda.synchronize()
        log("bounded mixed solve: %d iterations, %d reliable updates" % (it, nrel))
        return 0

    # FP64 reference solve: time to solution of the plain FP64 GPU path, and
    # the solution the mixed solver is compared with
    fp64 = {}
    if args.solver != "f64":
        solve_f64()
        torch.cuda.synchronize()
        t0 = torch.cuda.Event(enable_timing=True); t1 = torch.cuda.Event(enable_timing=True)
        t0.record(stream)
        it64, _, tr64 = solve_f64()
        t1.record(stream)
        torch.cuda.synchronize()
        fp64 = {"ms": t0.elapsed_time(t1), "iters": it64, "true_rel": tr64 / bnorm2, "x": x.clone()}
        log("FP64 solve: %.1f ms, %d iterations, true |r|^2/|b|^2 = %.3e"
            % (fp64["ms"], it64, tr64 / bnorm2))
        g.set_link_recon(18)
        t0.record(stream)
        it18, _, tr18 = solve_f64()
        t1.record(stream)
        torch.cuda.synchronize()
        g.set_link_recon(12)
        fp64["ms18"], fp64["iters18"], fp64["true_rel18"] = t0.elapsed_time(t1), it18, tr18 / bnorm2
        log("FP64 solve, 18-real links: %.1f ms, %d iterations, true |r|^2/|b|^2 = %.3e"
            % (fp64["ms18"], it18, tr18 / bnorm2))

    for _ in range(args.warmup):
        it, nrel, tr = solve()
        log("warmup solve: %d iterations, %d reliable updates, true |r|^2/|b|^2 = %.3e"
            % (it, nrel, tr / bnorm2))
    torch.cuda.synchronize()
    times, iters, trs, nrels = [], [], [], []
    for _ in range(args.steps):
        torch.cuda.synchronize()
        s0, s1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s0.record(stream)
        it, nrel, tr = solve()
        s1.record(stream)
        torch.cuda.synchronize()
        times.append(s0.elapsed_time(s1))
        iters.append(it)
        trs.append(tr)
        nrels.append(nrel)
    ms = sum(times) / len(times)
    true_rel = max(trs) / bnorm2
    sol_err = None
    if fp64:
        sol_err = float(torch.linalg.vector_norm(x - fp64["x"]) / torch.linalg.vector_norm(fp64["x"]))
    log("%s solve: %.1f ms, %d iterations, %d reliable updates, true |r|^2/|b|^2 = %.3e, "
        "|x-x64|/|x64| = %s" % (args.solver, ms, iters[0], nrels[0], true_rel, sol_err))
    # every solve must reach its bound: a missed residual fails the run (the
    # line is still printed, with the failures named in it)
    failures = []
    if true_rel > 1e-20:
        failures.append("%s solve: true |r|^2/|b|^2 = %.3e > 1e-20" % (args.solver, true_rel))
    if fp64 and fp64["true_rel"] > 1e-20:
        failures.append("FP64 solve: true |r|^2/|b|^2 = %.3e > 1e-20" % fp64["true_rel"])
    if fp64 and fp64["true_rel18"] > 1e-20:
        failures.append("FP64 solve (18-real links): true |r|^2/|b|^2 = %.3e > 1e-20" % fp64["true_rel18"])

    # the dominant kernel of the mixed solve: the 16-bit hopping kernel, timed in
    # isolation with HIP events on the context stream
    roof16 = None
    if args.solver == "mixed16":
        ms16 = g.time_dslash_lp(b, "f16", reps=args.dslash_reps)
        b16 = DSLASH16_CLINV_BYTES_PER_SITE * vh
        gbs16 = b16 / (ms16 * 1e-3) / 1e9
        log("16-bit dslash (A^-1 D): %.4f ms/launch, %.1f GB/s algorithmic" % (ms16, gbs16))
        traffic16, traffic16_src = measured_traffic(L, "f16")
        roof16 = {"bound": "hbm", "achieved": gbs16, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                  "frac": gbs16 / HBM_PEAK_GBS, "traffic": traffic16, "traffic_source": traffic16_src,
                  "kernel": "k_dslash<SF16, SF16, false, EPI_CLINV> (16-bit hopping matrix with "
                            "the A^-1 epilogue; 4 such launches per inner iteration)",
                  "bytes_per_launch": b16, "ms_per_launch": ms16,
                  "GFlops_hopping": DSLASH_FLOPS_PER_SITE * vh / (ms16 * 1e-3) / 1e9,
                  "note": "no unit saturated at 32^3x64: VALU 60 %, texture addresser 71 %, "
                          "HBM 5.7 TB/s (profiles/dslash_counters_32x32x32x64.md)"}

    # precision comparison (FP32 inner, then 16-bit storage) at the reliable-update
    # settings the precision configuration prescribes: update every 100 inner
    # iterations or when the residual drops by 1e-2; each against the FP64 solve
    sweep = None
    if not args.no_sweep and fp64:
        sweep = {}
        for name, prec, delta, mi in (("f32_delta1e-2_every100", "f32", 1e-2, 100),
                                      ("f16_delta1e-2_every100", "f16", 1e-2, 100),
                                      ("f32_delta1e-1_every1000", "f32", 0.1, 1000),
                                      ("f16_delta1e-1_every1000", "f16", 0.1, 1000)):
            x.zero_()
            torch.cuda.synchronize()
            q0, q1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            q0.record(stream)
            it_s, nrel_s, tr_s = g.cg_mixed_d("mtdagmt", x, b, kappa, rest=rest, maxiter=40000,
                                              precision=prec, delta=delta, max_inner=mi)
            q1.record(stream)
            torch.cuda.synchronize()
            ms_s = q0.elapsed_time(q1)
            sweep[name] = {
                "s": ms_s / 1e3, "iterations": it_s, "reliable_updates": nrel_s,
                "true_residual_rel": tr_s / bnorm2,
                "solution_rel_error_vs_fp64": float(torch.linalg.vector_norm(x - fp64["x"])
                                                    / torch.linalg.vector_norm(fp64["x"])),
                "speedup_vs_fp64": fp64["ms"] / ms_s,
            }
            log("precision", name, json.dumps(sweep[name]))
            if tr_s / bnorm2 > 1e-20:
                failures.append("precision run %s: true |r|^2/|b|^2 = %.3e > 1e-20" % (name, tr_s / bnorm2))

    cpu = None
    if not args.no_cpu:
        try:
            cpu = cpu_baseline(g, b, kappa, csw, fp64.get("iters", iters[0]), args.cpu_iters)
            log("cpu baseline:", cpu)
        except Exception as exc:  # reported, never silently replaced
            log("cpu baseline failed:", exc)

    batch = None
    if not args.no_batch:
        g.close()
        batch = batched(args, torch, dev, stream)
        if batch["max_true_residual_rel"] > 1e-20:
            failures.append("batched solve: true |r|^2/|b|^2 = %.3e > 1e-20"
                            % batch["max_true_residual_rel"])

    cg_bytes = CG_ITER_BYTES_PER_SITE_12 * vh * (fp64.get("iters") or iters[0])
    traffic, traffic_src = measured_traffic(L)
    fp64_ms = fp64.get("ms", ms)
    line = {
        "metric": "CG time to |r|/|b|<=1e-10: mixed+batched vs FP64 GPU; D-slash HBM GB/s",
        "value": ms / 1e3,
        "unit": "s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"f64": "f64", "mixed32": "f32 inner / f64 reliable", "mixed16": "f16 storage + f32 arithmetic inner / f64 reliable"}[args.solver],
        "data": "synthetic (seeded Haar SU(3) + 5 APE sweeps, alpha %.2f; Gaussian source)" % args.alpha,
        "config": {
            "workload": "CG on M~^+M~ to |r|/|b|<=1e-10, clover-Wilson even-odd, %s" % "x".join(map(str, L)),
            "lattice": list(L), "kappa": kappa, "csw": csw, "plaquette": round(plaq, 6),
            "solver": args.solver, "iterations": iters[0], "reliable_updates": nrels[0],
            "true_residual_rel": true_rel, "solution_rel_error_vs_fp64": sol_err,
            "delta": args.delta, "max_inner": args.max_inner,
            "parallelism": "single GPU",
        },
        "fp64_cg_s": fp64_ms / 1e3,
        "fp64_cg_iterations": fp64.get("iters", iters[0]),
        "speedup_vs_fp64": fp64_ms / ms,
        "fp64_cg_algorithmic_GBs": cg_bytes / (fp64_ms * 1e-3) / 1e9,
        "fp64_cg_link_reals": 12,
        "fp64_cg_ms_per_iteration": fp64_ms / (fp64.get("iters") or iters[0]),
        "fp64_cg_18real_s": fp64.get("ms18", float("nan")) / 1e3,
        "fp64_cg_18real_iterations": fp64.get("iters18"),
        "fp64_cg_18real_algorithmic_GBs": (CG_ITER_BYTES_PER_SITE_18 * vh * fp64["iters18"]
                                           / (fp64["ms18"] * 1e-3) / 1e9) if fp64 else None,
        "dslash_fp64_ms": ds_ms,
        "dslash_fp64_GBs": ds_gbs,
        "dslash_fp64_GFlops": DSLASH_FLOPS_PER_SITE * vh / (ds_ms * 1e-3) / 1e9,
        "roofline": {
            "bound": "hbm",
            "achieved": ds_gbs,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": ds_gbs / HBM_PEAK_GBS,
            "traffic": traffic,
            "traffic_source": traffic_src,
            "kernel": "k_dslash<SF64, false, EPI_PLAIN> (FP64 hopping matrix, one parity)",
            "bytes_per_launch": ds_bytes,
        },
        "roofline_mixed16": roof16,
        "cpu_baseline": cpu,
        "precision_comparison": sweep,
        "batched": batch,
    }
    if failures:
        line["residual_check"] = {"failed": failures}
    print(json.dumps(line), flush=True)
    g.close()
    for msg in failures:
        log("FAILED:", msg)
    return 1 if failures else 0


if __name__ == "__main__":
    sys.exit(main())
