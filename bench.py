#!/usr/bin/env python3
"""Collision-operator benchmark: Q(f) evaluations per second at a 32^3 velocity grid.

One step = one batched evaluation of Q over every point of the workload (the
``collide`` of one RK stage): 4096 spatial points of the lid-driven-cavity
shape (16x16 quads, p=3: 16 solution points x 256 elements), Nv=32 on
[-6,6]^3, M=12 directions, Nrho=16 radial points, omega=0.81.  The timed
call is the drop-in entry point on the solver's AoSoA distribution register
(dgfs_vhs_eval, what fs_batch calls); the contiguous entry point is timed
beside it.  The headline path computes transforms and products in FP32 and
projects Q onto the five collision invariants in FP64; the plain FP64 path
is measured in the same run, as are the FP32-vs-FP64 errors with and without
the projection.  States are synthetic (seeded bimodal and anisotropic
Maxwellians, density 1) generated on the device, so the timed region starts
with the inputs resident in HBM.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W]
Prints one JSON line; the full record, with its threshold tables, goes to stderr.
"""
import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, "dgfs-be-solver_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

METRIC = "Q(f) evals/s at 32^3 v-grid; FP32/surrogate vs FP64 spectral at ≤1e-3 rel L2"
HBM_PEAK = 8.0e12          # B/s, MI355X HBM3E
FP32_PEAK = 157.3e12       # FLOP/s, MI355X FP32 (vector and dense matrix)
FP64_PEAK = 78.6e12


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--points", type=int, default=4096)
    ap.add_argument("--nupts", type=int, default=16,
                    help="solution points per element of the AoSoA register (16: quads at p = 3)")
    ap.add_argument("--nv", type=int, default=32)
    ap.add_argument("--nrho", type=int, default=16)
    ap.add_argument("--M", type=int, default=12)
    ap.add_argument("--L", type=float, default=6.0)
    ap.add_argument("--omega", type=float, default=0.81)
    ap.add_argument("--fp64-steps", type=int, default=3)
    ap.add_argument("--cpu-points", type=int, default=16)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-fp64", action="store_true")
    ap.add_argument("--rhs-steps", type=int, default=3,
                    help="timed SSP-RK2 steps of the 16x16 p=3 cavity (two RHS evaluations each); 0 skips")
    ap.add_argument("--sur-train", type=int, default=131072,
                    help="synthetic near-equilibrium training states of the learned surrogate, besides "
                         "the cavity snapshots (0 skips the surrogate section)")
    ap.add_argument("--sur-epochs", type=int, default=20)
    ap.add_argument("--sur-cavity-snaps", type=int, default=16,
                    help="training snapshots (4096 states each) from a run of the lid-driven cavity; "
                         "the state one interval later is the evaluation workload (0 skips the cavity)")
    ap.add_argument("--sur-cavity-every", type=int, default=12,
                    help="SSP-RK2 steps between cavity snapshots")
    ap.add_argument("--sur-threshold", type=float, default=0.05)
    ap.add_argument("--sur-tol", type=float, default=1e-3,
                    help="target relative L2 error of the sampled spectral check")
    ap.add_argument("--sur-threshold-hi", type=float, default=1e-3,
                    help="fallback also where the share of f's norm in modes of degree >= 4 exceeds this")
    ap.add_argument("--algorithm", type=int, default=0,
                    help="gain kernel of the FP32 path: 0 automatic, 1 multi-pass, 2 register-resident, "
                         "3 register-resident with in-kernel Nyquist planes")
    ap.add_argument("--groups", type=int, default=0,
                    help="radial groups per point of the FP32 gain launch (0: the library's choice)")
    ap.add_argument("--pair-points", type=int, default=1024,
                    help="second batch of the batching workload, evaluated with the first in one paired "
                         "call (0 skips the section)")
    ap.add_argument("--pair-nv", type=int, default=24)
    ap.add_argument("--pair-steps", type=int, default=3)
    ap.add_argument("--pair-cpu-points", type=int, default=2,
                    help="points per grid checked against the FP64 oracle")
    ap.add_argument("--vss-points", type=int, default=2048,
                    help="two-species mixture batch (0 skips): points per species")
    ap.add_argument("--vss-steps", type=int, default=3)
    ap.add_argument("--vss-nv", type=int, default=24)
    ap.add_argument("--vss-L", type=float, default=6.0)
    ap.add_argument("--vss-cpu-points", type=int, default=8)
    ap.add_argument("--vss-algorithm", type=int, default=0,
                    help="two-species gain kernel (0 automatic, 1 multi-pass, 4 register-resident, "
                         "6 packed isotropic)")
    ap.add_argument("--calibrate-copy-mib", type=int, default=0,
                    help="before the bench, run 3 plain device copies (torch elementwise "
                         "multiply by 1) of this many MiB, so that a counter run sees a "
                         "kernel of known traffic next to the measured ones")
    return ap.parse_args()


def calibrate_copy(mib, device):
    """Three launches of a plain elementwise copy reading and writing `mib` MiB
    each; a FETCH_SIZE / WRITE_SIZE counter run divides what it reads for
    them by mib*1024 KiB to get the counter's scale."""
    import torch
    n = mib * (1 << 20) // 8
    a = torch.ones(n, dtype=torch.float64, device=device)
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    for _ in range(3):
        torch.mul(a, 1.0, out=b)
    torch.cuda.synchronize()
    print(f"# copy calibration: 3 x {mib} MiB read + {mib} MiB written", file=sys.stderr, flush=True)
    del a, b
    torch.cuda.empty_cache()


def bench_rhs(args, dev):
    """RHS evaluations/s of the lid-driven cavity: 16x16 quads, p = 3 (4096
    solution points), Nv = 32 on [-6, 6]^3, M = 12, Nrho = 16, omega = 0.81,
    Kn = 0.05, lid speed 0.3; FP32 collision operator with FP64 projection.
    One RHS evaluation = collide over all points + advection of all velocity
    columns + boundary update; an SSP-RK2 step is two.  Timed as HIP-graph
    replays of whole steps (one launch per step) and as eager steps."""
    import numpy as np
    import torch

    from dgfs_hip.backend import HIPBackend
    from dgfs_hip.cases import cavity_cfg
    from dgfs_hip.integrators.graphs import GraphStepper
    from dgfs_hip.integrators.steppers import get_stepper
    from dgfs_hip.mesh import rect_quads
    from dgfs_hip.solvers.dgfs.system import DGFSSystem

    cfg = cavity_cfg(Nv=args.nv, L=args.L, Nrho=args.nrho, M=args.M, Kn=0.05, omega=args.omega, order=3,
                     ulid=0.3, precision="single", project=True)
    be = HIPBackend(cfg, own_stream=True)
    mesh = rect_quads(16, 16, 0.0, 1.0, 0.0, 1.0)
    sysm = DGFSSystem(be, mesh, cfg, 3)
    # SSP-RK2 with the p = 3 FR operator needs a step well below the unit-CFL
    # step to stay bounded over long runs; the throughput does not depend on it
    dt = 0.05 * sysm.unit_cfl_dt
    st = get_stepper("dgfs-tvd-rk2", be, sysm, dt)
    gs = GraphStepper(st)
    out = {"workload": "cavity 16x16 quads p=3 (4096 points), Nv=32, M=12, Nrho=16, SSP-RK2, "
                       "FP32 collision + FP64 projection",
           "points": sysm.ele.nupts * sysm.ele.neles}
    # eager step (also the graph warm-up), then capture + first replay
    for _ in range(2):
        st._idxcurr = gs.step(st.tcurr, dt)
        st.tcurr += dt
    be.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.rhs_steps):
        st._idxcurr = gs.step(st.tcurr, dt)
        st.tcurr += dt
    be.synchronize()
    tg = time.perf_counter() - t0
    t0 = time.perf_counter()
    for _ in range(args.rhs_steps):
        st._idxcurr = st.step(st.tcurr, dt)
        st.tcurr += dt
    be.synchronize()
    te = time.perf_counter() - t0
    # share of the collision operator in one eager RHS evaluation
    op = sysm.sm.op
    op.set_timing(True)
    st._idxcurr = st.step(st.tcurr, dt)
    be.synchronize()
    tim = op.get_timing()
    op.set_timing(False)
    coll_ms = sum(v[0] for v in tim.values()) / 2.0
    # the advection and boundary kernels of one RHS evaluation alone, timed
    # with events on the solver's stream
    vmr = sysm.vm
    NvBS = vmr.NvBatchSize()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    be.synchronize()
    ev0.record(be._stream)
    for batch in range(vmr.NvBatches()):
        sysm.updatebc(st.tcurr, st.soln_bank, 1, batch, batch * NvBS)
    for batch in range(vmr.NvBatches()):
        sysm.rhs(st.tcurr, st.soln_bank, 1, batch, batch * NvBS)
    ev1.record(be._stream)
    be.synchronize()
    fr_ms = ev0.elapsed_time(ev1)
    frb = fr_rhs_bytes(sysm)
    fr_total = float(sum(frb.values()))
    npts = out["points"]
    bq = algorithmic_bytes(vmr.Nv(), vmr.Nrho() * vmr.M(), 8)
    rhs_bytes = npts * bq + fr_total
    ms_rhs = 1e3 * tg / (2 * args.rhs_steps)
    out["roofline"] = {
        "bound": "hbm", "unit": "GB/s", "peak": HBM_PEAK / 1e9,
        "achieved": rhs_bytes / (ms_rhs / 1e3) / 1e9,
        "frac": rhs_bytes / (ms_rhs / 1e3) / HBM_PEAK,
        "bytes_per_rhs": rhs_bytes,
        "collision_bytes_per_rhs": npts * bq,
        "advection_bytes_per_rhs": fr_total,
        "advection_bytes_by_kernel": frb,
        "advection_ms_per_rhs": fr_ms,
        "advection_achieved_gbps": fr_total / (fr_ms / 1e3) / 1e9,
        "advection_frac": fr_total / (fr_ms / 1e3) / HBM_PEAK,
        "note": "RHS bytes = points x B_Q + the advection and boundary kernels' bytes; B_Q prices the "
                "reference dataflow's transforms crossing HBM (the collision kernels keep them on chip), "
                "so frac may exceed 1; advection_frac is the HBM fraction of the FR kernels alone",
    }
    out.update({
        "rhs_evals_per_s": 2 * args.rhs_steps / tg,
        "rhs_evals_per_s_eager": 2 * args.rhs_steps / te,
        "ms_per_rhs_graph": 1e3 * tg / (2 * args.rhs_steps),
        "ms_per_rhs_eager": 1e3 * te / (2 * args.rhs_steps),
        "collide_ms_per_rhs": coll_ms,
        "graph_nodes_per_step": gs.nodes,
        "steps": args.rhs_steps,
    })
    f = sysm.eles_scal_upts_full[st.soln_bank].get()
    out["finite"] = bool(np.isfinite(f).all())
    gs.close()
    del sysm, be
    torch.cuda.empty_cache()
    return out


def fr_rhs_bytes(sysm):
    """Algorithmic HBM bytes of the advection and boundary kernels of one RHS
    evaluation over all velocity batches: per operator product
    (k + m + [beta != 0] m) ncol s + m k s, per pointwise kernel the arrays it
    reads and writes once (the interface kernels read and write both sides'
    flux-point states).  Returns {kernel: bytes}."""
    ele, vm = sysm.ele, sysm.vm
    s = 8
    reg = ele.scal_upts[0]
    ncol, nparr = reg.ncol, reg.ncol // ele.nvars
    nupts, nfpts, ndims, nvars = ele.nupts, ele.nfpts, ele.ndims, ele.nvars

    def mul(m, k, beta):
        return ((k + m + (m if beta else 0)) * ncol + m * k) * s
    per = {
        "mul M0 (disu, rhs and updatebc)": 2 * mul(nfpts, nupts, False),
        "tflux": (nupts + ndims * nupts) * ncol * s + ndims * ndims * nupts * nparr * s,
        "mul M1-M3*M2 (tdivtpcorf)": mul(nupts, ndims * nupts, False),
        "intcflux": 4 * sysm.iint.ninterfpts * nvars * s,
        "bccflux": sum(2 * b.ninterfpts * nvars * s for b in sysm.bcints),
        "bccupdate": sum(b.ninterfpts * nvars * s for b in sysm.bcints if getattr(b, "updates", False)),
        "mul M3 (tdivtconf, beta = 1)": mul(nupts, nfpts, True),
        "negdivconf": 2 * nupts * ncol * s + nupts * nparr * s,
    }
    return {k: v * vm.NvBatches() for k, v in per.items()}


def vss_bytes(nv, K, S, c):
    """Algorithmic HBM bytes of one mixture point in the reference dataflow
    (dgfsbi/scattering.py:259-330): per ordered pair 3K transforms (two
    inverse, one forward per (radial, direction) item), per species the
    forward transform of f_p and the inverse of its gain and loss, each
    reading and writing one complex cube of c bytes per value."""
    n = nv ** 3
    return 2 * c * n * (3 * K * S * S + 3 * S)


def bench_vss(args, dev, stream):
    """Two-species VSS mixture (mass ratio 2.1, omega 0.81 / 0.805 / 0.80,
    VHS alpha = 1) on one Nv^3 grid: FP32 + FP64 mixture projection against
    the plain FP64 path, per-species error, mixture conservation."""
    import numpy as np
    import torch
    from dgfs_hip.solvers.dgfsbi.scattering import VSSOperator
    from dgfs_hip.solvers.dgfsbi.velocitymesh import DGFSBiVelocityMesh
    from dgfs_hip.sphericaldesign import get_sphquadrule
    nv, L, Nrho, M, Mpre, P = args.vss_nv, args.vss_L, 12, 12, 24, args.vss_points
    masses = (1.0, 2.1)
    omegas = np.array([[0.81, 0.805], [0.805, 0.80]])
    vm = DGFSBiVelocityMesh.from_params(None, nv, L, Nrho, M, masses)
    S, K = 2, Nrho * M
    gamma, eta, prefac = 2.0 * (1.0 - omegas), np.zeros((S, S)), np.ones((S, S))
    szpre = get_sphquadrule("symmetric", npts=Mpre).pts
    cv = torch.as_tensor(vm.cv(), device=dev)
    g = torch.Generator(device="cpu").manual_seed(7)
    fs = []
    for p, m in enumerate(vm.masses()):
        u = (torch.rand((P, 3, 1, 2), generator=g, dtype=torch.float64) * 2 - 1).to(dev)
        T = (0.6 + 1.2 * torch.rand((P, 1, 2), generator=g, dtype=torch.float64)).to(dev)
        c2 = ((cv[None, :, :, None] - u) ** 2).sum(1)                 # (P, n, 2)
        mx = (m / (math.pi * T)) ** 1.5 * torch.exp(-m * c2 / T)
        fs.append((0.5 * mx[..., 0] + 0.5 * mx[..., 1]).contiguous())
    Qs32 = [torch.empty_like(f) for f in fs]
    ptr = lambda a: [x.data_ptr() for x in a]
    op32 = VSSOperator(nv, Nrho, M, vm.L(), vm.sw(), vm.cw(), vm.qz(), vm.qw(), vm.sz(), szpre,
                       vm.masses(), gamma, eta, prefac, precision=32, project=True)
    if args.vss_algorithm:
        op32.set_algorithm(args.vss_algorithm)
    op32.eval_contig(ptr(fs), ptr(Qs32), P, stream)
    torch.cuda.synchronize()
    op32.set_timing(True)
    t0 = time.perf_counter()
    for _ in range(args.vss_steps):
        op32.eval_contig(ptr(fs), ptr(Qs32), P, stream)
    torch.cuda.synchronize()
    w32 = time.perf_counter() - t0
    tim = op32.get_timing()
    cfgv = op32.get_config()
    op32.set_timing(False)
    gain_ms, gain_n = tim["gain"]
    algo = op32.get_algorithm()
    kname = {4: f"k_vss_gain_rr1<float,{nv}>", 5: f"k_vss_gain_rr1_iso<float,{nv}>",
             6: f"k_vss_gain_rr1_isop<float,{nv}>",
             7: f"k_vss_gain_slab<float,{nv}> + k_vss_xfwd<float,{nv}>"}.get(algo, f"k_vss_gain<float,{nv}>")
    bq = vss_bytes(nv, K, S, 8)
    achieved = bq * P * args.vss_steps / (gain_ms / 1e3)
    # HBM bytes per launch from the committed counter runs, scaled to this batch
    tr = read_traffic({4: f"vss_gain_rr1_fp32_n{nv}_traffic.json",
                       5: f"vss_gain_rr1_iso_fp32_n{nv}_traffic.json",
                       6: f"vss_gain_rr1_isop_fp32_n{nv}_traffic.json",
                       7: f"vss_gain_slab_fp32_n{nv}_traffic.json"}.get(algo, ""))
    traffic = (tr["bytes_per_dispatch"] * P * args.vss_steps / max(gain_n, 1) / tr["points_per_dispatch"]
               if tr else None)
    out = {
        "workload": f"two-species VSS mixture: {P} points, Nv={nv} on [-{L:g},{L:g}]^3, M={M}, Nrho={Nrho}, "
                    f"Mpre={Mpre}, masses 1 / 2.1, omega 0.81 / 0.805 / 0.80, bimodal species states",
        "unit": "mixture points/s (every species' Q_p at one point)",
        "value": P * args.vss_steps / w32,
        "pair_evals_per_s": S * S * P * args.vss_steps / w32,
        "ms_per_step": 1e3 * w32 / args.vss_steps,
        "dtype": "f32+fp64-projection",
        "kernel_ms_per_step": {k: v[0] / args.vss_steps for k, v in tim.items()},
        "config": cfgv,
        "roofline": {"bound": "hbm", "kernel": kname, "achieved": achieved / 1e9,
                     "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": achieved / HBM_PEAK,
                     "algorithmic_bytes_per_point": bq,
                     "avg_launch_ms": gain_ms / max(gain_n, 1), "traffic": traffic,
                     "note": "reference dataflow with every transform crossing HBM once; the kernel "
                             "keeps them in LDS/registers"},
    }
    op32.close()
    op64 = VSSOperator(nv, Nrho, M, vm.L(), vm.sw(), vm.cw(), vm.qz(), vm.qw(), vm.sz(), szpre,
                       vm.masses(), gamma, eta, prefac, precision=64, project=False)
    Qs64 = [torch.empty_like(f) for f in fs]
    op64.eval_contig(ptr(fs), ptr(Qs64), P, stream)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    op64.eval_contig(ptr(fs), ptr(Qs64), P, stream)
    torch.cuda.synchronize()
    w64 = time.perf_counter() - t0
    op64.close()
    op64p = VSSOperator(nv, Nrho, M, vm.L(), vm.sw(), vm.cw(), vm.qz(), vm.qw(), vm.sz(), szpre,
                        vm.masses(), gamma, eta, prefac, precision=64, project=True)
    Qs64p = [torch.empty_like(f) for f in fs]
    op64p.eval_contig(ptr(fs), ptr(Qs64p), P, stream)
    torch.cuda.synchronize()
    op64p.close()
    out["fp64_plain"] = {"value": P / w64, "ms_per_step": 1e3 * w64}
    out["fp32_speedup_vs_fp64"] = out["value"] / out["fp64_plain"]["value"]
    out["fp32_vs_fp64_rel_l2_per_species"] = [
        float(torch.linalg.norm(a - b) / torch.linalg.norm(b)) for a, b in zip(Qs32, Qs64p)]
    # mixture invariants of the FP32 result: species masses, total momentum, total energy
    w = vm.cw()
    mass = max(float(((q.sum(1) * w).abs() / (q.abs().sum(1) * w)).max()) for q in Qs32)
    scale = sum(m * q.abs().sum(1) * w for m, q in zip(vm.masses(), Qs32))
    mom = sum(m * (q @ cv.T) * w for m, q in zip(vm.masses(), Qs32))            # (P, 3)
    en = sum(m * (q @ (cv ** 2).sum(0)) * w for m, q in zip(vm.masses(), Qs32))
    out["conservation_after_projection_max_rel"] = {
        "species_mass": mass, "momentum": float((mom.abs().max(1).values / scale).max()),
        "energy": float((en.abs() / scale).max())}
    if args.vss_cpu_points > 0 and not args.no_cpu:
        from oracle import vss as V
        ov = V.BiVelocityMesh(nv, L, Nrho, M, masses)
        pairs = [(p, q) for p in range(S) for q in range(S)]
        orc = V.VSSOracle(ov, {k: gamma[k] for k in pairs}, {k: 0.0 for k in pairs},
                          {k: 1.0 for k in pairs}, szpre)
        k = args.vss_cpu_points
        sample = [f[:k].cpu().numpy() for f in fs]
        t0 = time.perf_counter()
        qo = orc.q(sample)
        tc = time.perf_counter() - t0
        out["cpu_baseline"] = {"value": k / tc, "unit": out["unit"], "cores": 1, "kind": "port",
                               "sample": f"FP64 numpy/scipy.fft restatement of the reference dataflow on "
                                         f"the first {k} point(s) of the same batch, one core"}
        out["fp64_gpu_vs_oracle_rel_l2"] = [
            float(np.linalg.norm(q64[:k].cpu().numpy() - o) / np.linalg.norm(o)) for q64, o in zip(Qs64, qo)]
    del Qs32, Qs64, Qs64p, fs
    return out


def bimodal_states(vm, npts, seed, device):
    """Seeded bimodal Maxwellians 1/2 M(1, u1, T1) + 1/2 M(1, u2, T2) with the
    means uniform in the unit ball and T ~ U[0.5, 2], renormalised to density 1
    on the grid (the second batch of the precision + batching workload)."""
    import numpy as np
    import torch
    rng = np.random.default_rng(seed)
    cv = torch.as_tensor(vm.cv(), device=device)
    out = torch.empty((npts, vm.vsize()), dtype=torch.float64, device=device)
    for i in range(npts):
        f = torch.zeros(vm.vsize(), dtype=torch.float64, device=device)
        for _ in range(2):
            d = rng.normal(size=3)
            u = d / np.linalg.norm(d) * rng.uniform(0, 1) ** (1 / 3)
            T = rng.uniform(0.5, 2.0)
            ut = torch.as_tensor(u, device=device).view(3, 1)
            f += 0.5 * torch.exp(-((cv - ut) ** 2).sum(0) / T) / (math.pi * T) ** 1.5
        out[i] = f / (f.sum() * vm.cw())
    return out


def bench_pair(args, dev, stream):
    """The batching workload: the 4096 cavity-shape points at 32^3 and a second
    batch of 1024 homogeneous bimodal points at 24^3 (same box, M, Nrho,
    omega; FP32 + FP64 projection) evaluated by one paired call, in which the
    two register-resident gains run back to back (their kernels need different
    workgroup sizes); against the two batches evaluated by separate calls, with
    per-grid errors against the FP64 oracle on a sample.  The one-launch form
    (both grids' multi-pass gain items in one persistent launch) is timed
    beside it."""
    import numpy as np
    import torch
    from dgfs_hip.solvers.dgfs.scattering import VHSOperator
    from dgfs_hip.solvers.dgfs.velocitymesh import DGFSVelocityMesh
    gamma = 2.0 * (1.0 - args.omega)
    vma = DGFSVelocityMesh.from_params(None, args.nv, args.L, args.nrho, args.M)
    vmb = DGFSVelocityMesh.from_params(None, args.pair_nv, args.L, args.nrho, args.M)
    Pa, Pb = args.points, args.pair_points
    fa = make_states(vma, Pa, seed=0, device=dev)
    fb = bimodal_states(vmb, Pb, seed=5, device=dev)
    Qa, Qb = torch.empty_like(fa), torch.empty_like(fb)
    opa = VHSOperator.from_mesh(vma, gamma, 1.0, precision=32, project=True)
    opb = VHSOperator.from_mesh(vmb, gamma, 1.0, precision=32, project=True)

    def sep():
        opa.eval_contig(fa.data_ptr(), Qa.data_ptr(), Pa, stream)
        opb.eval_contig(fb.data_ptr(), Qb.data_ptr(), Pb, stream)

    def pair():
        opa.eval_pair(fa.data_ptr(), Qa.data_ptr(), Pa, opb, fb.data_ptr(), Qb.data_ptr(), Pb, stream)

    out = {"workload": f"{Pa} points at {args.nv}^3 (cavity-shape bimodal / anisotropic states) + {Pb} "
                       f"homogeneous bimodal points at {args.pair_nv}^3, both on [-{args.L:g},{args.L:g}]^3, "
                       f"M={args.M}, Nrho={args.nrho}, omega={args.omega}, FP32 + FP64 projection",
           "unit": "Q(f) evals/s (both grids)"}
    for name, fn in (("separate", sep), ("pair", pair)):
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.pair_steps):
            fn()
        torch.cuda.synchronize()
        w = (time.perf_counter() - t0) / args.pair_steps
        out[name] = {"value": (Pa + Pb) / w, "ms_per_step": 1e3 * w}
    out["value"] = out["pair"]["value"]
    out["algorithms"] = [opa.get_algorithm(), opb.get_algorithm()]
    # the literal one-launch form: multi-pass gain items of both grids in one
    # persistent launch
    opa.set_algorithm(1)
    opb.set_algorithm(1)
    pair()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    pair()
    torch.cuda.synchronize()
    w = time.perf_counter() - t0
    out["one_launch_multipass"] = {"value": (Pa + Pb) / w, "ms_per_step": 1e3 * w}
    opa.set_algorithm(0)
    opb.set_algorithm(0)
    pair()
    torch.cuda.synchronize()
    Qa_p, Qb_p = Qa.clone(), Qb.clone()
    sep()
    torch.cuda.synchronize()
    out["pair_equals_separate_bitwise"] = bool(torch.equal(Qa_p, Qa) and torch.equal(Qb_p, Qb))
    if not args.no_cpu and args.pair_cpu_points > 0:
        from oracle import vhs as O
        k = args.pair_cpu_points
        errs = {}
        for nv, f, Q in ((args.nv, fa, Qa_p), (args.pair_nv, fb, Qb_p)):
            ov = O.VelocityMesh(nv, args.L, args.nrho, args.M)
            ref = O.project_invariants(ov, O.VHSOracle(ov, gamma, 1.0).q(f[:k].cpu().numpy(), workers=16))
            errs[f"{nv}^3"] = float(np.linalg.norm(Q[:k].cpu().numpy() - ref) / np.linalg.norm(ref))
        out["fp32_vs_fp64_oracle_rel_l2_per_grid"] = errs
        out["oracle_sample_points_per_grid"] = k
    opa.close()
    opb.close()
    del fa, fb, Qa, Qb, Qa_p, Qb_p
    return out


def mild_states(vm, npts, seed, device):
    """Seeded anisotropic Gaussians (axis temperatures within a factor 1.5 of
    each other) and bimodal Maxwellians (half-separation |u| <= 0.3): the
    part of the bimodal / anisotropic families close to equilibrium."""
    import numpy as np
    import torch
    rng = np.random.default_rng(seed)
    cv = torch.as_tensor(vm.cv(), device=device)
    out = torch.empty((npts, vm.vsize()), dtype=torch.float64, device=device)
    for i in range(npts):
        u0 = torch.as_tensor(rng.uniform(-0.4, 0.4, 3), device=device).view(3, 1)
        rho = rng.uniform(0.6, 1.4)
        if i % 2 == 0:
            T = rng.uniform(0.8, 1.2) * np.exp(rng.uniform(-0.2, 0.2, 3))
            Tt = torch.as_tensor(T, device=device).view(3, 1)
            f = torch.exp(-((cv - u0) ** 2 / Tt).sum(0)) / (math.pi ** 1.5 * math.sqrt(T.prod()))
        else:
            d = rng.normal(size=3)
            d *= rng.uniform(0, 0.3) / np.linalg.norm(d)
            dv = torch.as_tensor(d, device=device).view(3, 1)
            T = rng.uniform(0.7, 1.3, 2)
            f = (0.5 * torch.exp(-((cv - u0 - dv) ** 2).sum(0) / T[0]) / (math.pi * T[0]) ** 1.5
                 + 0.5 * torch.exp(-((cv - u0 + dv) ** 2).sum(0) / T[1]) / (math.pi * T[1]) ** 1.5)
        out[i] = rho * f / (f.sum() * vm.cw())
    return out


def near_equilibrium_states(vm, npts, seed, device, eps_range=(1e-3, 0.3), frac_far=0.05, frac_mild=0.0):
    """Seeded states of a low-Knudsen flow field: Maxwellians with random
    density, velocity and temperature carrying a Chapman-Enskog-like heat-flux
    and shear perturbation whose amplitude eps is log-uniform in eps_range
    (most points near equilibrium, a tail far from it), plus a fraction
    frac_far of bimodal / anisotropic states (the make_states recipe) and a
    fraction frac_mild of mild ones (mild_states)."""
    import numpy as np
    import torch
    rng = np.random.default_rng(seed)
    cv = torch.as_tensor(vm.cv(), device=device)
    out = torch.empty((npts, vm.vsize()), dtype=torch.float64, device=device)
    nfar = int(round(frac_far * npts))
    nmild = int(round(frac_mild * npts))
    if nfar:
        out[:nfar] = make_states(vm, nfar, seed + 1, device)
    if nmild:
        out[nfar:nfar + nmild] = mild_states(vm, nmild, seed + 2, device)
    # the perturbed Maxwellians, a chunk of points at a time
    i0, chunk = nfar + nmild, 512
    while i0 < npts:
        k = min(chunk, npts - i0)
        u = rng.uniform(-0.4, 0.4, (k, 3))
        T = rng.uniform(0.7, 1.4, k)
        rho = rng.uniform(0.6, 1.4, k)
        q = rng.normal(size=(k, 3))
        S = rng.normal(size=(k, 3, 3))
        S = S + S.transpose(0, 2, 1)
        S -= np.trace(S, axis1=1, axis2=2)[:, None, None] / 3 * np.eye(3)
        eps = np.exp(rng.uniform(math.log(eps_range[0]), math.log(eps_range[1]), k))
        ut, Tt, qt, St = (torch.as_tensor(x, device=device) for x in (u, T, q, S))
        c = (cv[None] - ut[:, :, None]) / torch.sqrt(Tt)[:, None, None]          # (k, 3, n)
        c2 = (c * c).sum(1)
        Sc = torch.einsum("kij,kjr->kir", St, c)
        phi = torch.as_tensor(eps, device=device)[:, None] * (
            0.4 * torch.einsum("ki,kir->kr", qt, c) * (c2 - 2.5) + 0.5 * (c * Sc).sum(1))
        out[i0:i0 + k] = (torch.as_tensor(rho, device=device) / (math.pi * Tt) ** 1.5)[:, None] \
            * torch.exp(-c2) * (1 + phi)
        i0 += k
    perm = torch.as_tensor(rng.permutation(npts), device=device)
    return out[perm].contiguous()


def cavity_snapshots(args, dev, nsnap, every, warm):
    """States of the lid-driven cavity of bench_rhs (16x16 quads, p = 3, 4096
    points; FP32 collision + FP64 projection; SSP-RK2 at 0.05 of the unit-CFL
    step, HIP-graph replays) as contiguous [point][velocity] FP64 device
    tensors, point = element * nupts + upt: after `warm` steps, then every
    `every` steps, nsnap snapshots in all.  Yields (tensor, step, time)."""
    import torch

    from dgfs_hip.backend import HIPBackend
    from dgfs_hip.cases import cavity_cfg
    from dgfs_hip.integrators.graphs import GraphStepper
    from dgfs_hip.integrators.steppers import get_stepper
    from dgfs_hip.mesh import rect_quads
    from dgfs_hip.solvers.dgfs.system import DGFSSystem

    cfg = cavity_cfg(Nv=args.nv, L=args.L, Nrho=args.nrho, M=args.M, Kn=0.05, omega=args.omega, order=3,
                     ulid=0.3, precision="single", project=True)
    be = HIPBackend(cfg, own_stream=True)
    sysm = DGFSSystem(be, rect_quads(16, 16, 0.0, 1.0, 0.0, 1.0), cfg, 3)
    dt = 0.05 * sysm.unit_cfl_dt
    st = get_stepper("dgfs-tvd-rk2", be, sysm, dt)
    gs = GraphStepper(st)
    nupts, neles, vsize = sysm.ele.nupts, sysm.ele.neles, sysm.vm.vsize()
    step = 0
    for k in range(nsnap):
        for _ in range(warm if k == 0 else every):
            st._idxcurr = gs.step(st.tcurr, dt)
            st.tcurr += dt
            step += 1
        be.synchronize()
        m = sysm.eles_scal_upts_full[st.soln_bank]
        nb = m.ncol // (vsize * 32)
        a = m.data[:, : m.ncol].view(nupts, nb, vsize, 32).permute(1, 3, 0, 2).reshape(nb * 32, nupts, vsize)
        f = a[:neles].reshape(neles * nupts, vsize).contiguous()
        torch.cuda.synchronize()
        yield f, step, st.tcurr
    gs.close()
    del sysm, be


def surrogate_eval(args, vm, sur, exact32, f, dev, stream):
    """Times and scores the surrogate with fallback on the states f [P][n]
    against the exact operators (FP32 for timing, FP64 for error)."""
    import torch

    from dgfs_hip.solvers.dgfs.scattering import VHSOperator

    P = f.shape[0]
    gamma = sur.gamma
    Q32 = torch.empty_like(f)
    exact32.eval_contig(f.data_ptr(), Q32.data_ptr(), P, stream)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    exact32.eval_contig(f.data_ptr(), Q32.data_ptr(), P, stream)
    torch.cuda.synchronize()
    t_ex32 = time.perf_counter() - t0
    del Q32
    op64 = VHSOperator.from_mesh(vm, gamma, 1.0, precision=64, project=True)
    Q64 = torch.empty_like(f)
    op64.eval_contig(f.data_ptr(), Q64.data_ptr(), P, stream)
    torch.cuda.synchronize()
    op64.close()
    mom = torch.empty((P, 8), dtype=torch.float64, device=dev)
    sur.encode(f, P, mom)
    torch.cuda.synchronize()
    ind = mom[:, 5]
    # a closure without the network at the same cost: BGK, nu (M[f] - f),
    # with the single nu that fits Q64 best over the points it would replace
    cvt = torch.as_tensor(vm.cv(), device=dev)
    Mf = mom[:, 0:1] / (math.pi * mom[:, 4:5]) ** 1.5 * torch.exp(
        -((cvt[0][None] - mom[:, 1:2]) ** 2 + (cvt[1][None] - mom[:, 2:3]) ** 2
          + (cvt[2][None] - mom[:, 3:4]) ** 2) / mom[:, 4:5])
    phi = torch.stack([torch.ones_like(cvt[0]), cvt[0], cvt[1], cvt[2], (cvt ** 2).sum(0)])
    Qs = torch.empty_like(f)
    per_thr = {}
    ind_hi = mom[:, 6]
    cases = [(args.sur_threshold, args.sur_threshold_hi), (0.02, 0.0), (0.05, 0.0), (0.1, args.sur_threshold_hi),
             (0.02, 1e-4), (0.005, 1e-4), (0.002, 0.0), (0.001, 0.0), (0.02, 1e-5), (0.005, 1e-5),
             (0.02, 3e-6), (0.02, 1e-6), (0.02, 3e-7)]
    seen = []
    for thr, thh in cases:
        if (thr, thh) in seen:
            continue
        seen.append((thr, thh))
        nfb = sur.eval_with_fallback(exact32, f, Qs, P, threshold=thr, threshold_hi=thh, stream=stream)
        torch.cuda.synchronize()
        reps = 3
        t0 = time.perf_counter()
        for _ in range(reps):
            nfb = sur.eval_with_fallback(exact32, f, Qs, P, threshold=thr, threshold_hi=thh, stream=stream)
        torch.cuda.synchronize()
        t_sur = (time.perf_counter() - t0) / reps
        mask = (ind <= thr) & ((ind_hi <= thh) if thh > 0 else torch.ones_like(ind, dtype=torch.bool))
        err = float(torch.linalg.norm(Qs - Q64) / torch.linalg.norm(Q64))
        err_pts = float(torch.linalg.norm((Qs - Q64)[mask]) / torch.linalg.norm(Q64[mask])) if mask.any() else 0.0
        d = (Mf - f)[mask]
        if mask.any():
            nu = float((d * Q64[mask]).sum() / (d * d).sum())
            err_bgk = float(torch.linalg.norm(nu * d - Q64[mask]) / torch.linalg.norm(Q64[mask]))
            Qb = Q64.clone()
            Qb[mask] = nu * d
            err_bgk_all = float(torch.linalg.norm(Qb - Q64) / torch.linalg.norm(Q64))
            del Qb
        else:
            err_bgk = err_bgk_all = 0.0
        cons = float((((Qs @ phi.T) * vm.cw()).abs() / (Qs.abs().sum(1, keepdim=True) * vm.cw())).max())
        per_thr[f"{thr:g}/{thh:g}"] = {
            "value": P / t_sur, "fallback_points": int(nfb), "fallback_rate": nfb / P,
            "rel_l2_vs_fp64": err, "rel_l2_vs_fp64_on_surrogate_points": err_pts,
            "rel_l2_bgk_best_nu_in_place_of_network": err_bgk_all,
            "rel_l2_bgk_best_nu_on_surrogate_points": err_bgk,
            "conservation_max_rel": cons,
        }
    # the sampled spectral check: a stratified sample of the surrogate
    # candidates is evaluated exactly and indicator-ranked bins fall back until
    # the estimated error of what the network keeps fits the target
    checked = {}
    for thr, thh in ((args.sur_threshold, args.sur_threshold_hi), (0.2, 0.0)):
        kw = dict(tol=args.sur_tol, threshold=thr, threshold_hi=thh, sample_frac=0.03, nbins=16, min_per_bin=4,
                  safety=0.7, seed=0)
        sur.eval_checked(exact32, f, Qs, P, stream=stream, **kw)
        torch.cuda.synchronize()
        reps = 3
        t0 = time.perf_counter()
        for _ in range(reps):
            stats = sur.eval_checked(exact32, f, Qs, P, stream=stream, **kw)
        torch.cuda.synchronize()
        t_chk = (time.perf_counter() - t0) / reps
        err = float(torch.linalg.norm(Qs - Q64) / torch.linalg.norm(Q64))
        checked[f"{thr:g}/{thh:g}"] = {
            "value": P / t_chk, "rel_l2_vs_fp64": err, "target": args.sur_tol,
            "fallback_rate": (stats["fallback_points"] + stats["sampled_points"]) / P, **stats}
    # the representation floor: the exact Q projected onto the network's
    # 8^3-mode span and decoded (what a perfect network would return), on the
    # points the head thresholds give to the surrogate
    _, _, y_true, mom_t = sur.make_dataset(f, Q64)
    Qf = torch.empty_like(f)
    sur.decode(y_true.contiguous(), mom_t, P, Qf, project=True)
    torch.cuda.synchronize()
    thr, thh = args.sur_threshold, args.sur_threshold_hi
    mask = (ind <= thr) & ((ind_hi <= thh) if thh > 0 else torch.ones_like(ind, dtype=torch.bool))
    floor_pts = float(torch.linalg.norm((Qf - Q64)[mask]) / torch.linalg.norm(Q64[mask])) if mask.any() else 0.0
    Qfl = Q64.clone()
    Qfl[mask] = Qf[mask]
    floor_all = float(torch.linalg.norm(Qfl - Q64) / torch.linalg.norm(Q64))
    del Qf, Qfl, y_true, mom_t
    head = per_thr[f"{args.sur_threshold:g}/{args.sur_threshold_hi:g}"]
    head = {**head, "rel_l2_representation_floor_on_surrogate_points": floor_pts,
            "rel_l2_representation_floor_overall": floor_all}
    ok = {k: v for k, v in per_thr.items() if v["rel_l2_vs_fp64"] <= 1e-3}
    ok.update({f"checked {k}": v for k, v in checked.items() if v["rel_l2_vs_fp64"] <= 1e-3})
    best = max(ok.items(), key=lambda kv: kv[1]["value"]) if ok else None
    out = {"points": P, "fallback_threshold": args.sur_threshold,
           "fastest_within_1e-3": ({"thresholds": best[0], **best[1]} if best else None),
           "sampled_spectral_check": checked,
           "fallback_threshold_high_modes": args.sur_threshold_hi, **head,
           "by_threshold": per_thr, "exact_fp32_evals_per_s_same_batch": P / t_ex32,
           "indicator_quantiles_10_50_90_99": [float(x) for x in torch.quantile(
               ind.float(), torch.tensor([0.1, 0.5, 0.9, 0.99], device=dev))]}
    del Mf, Q64, Qs
    return out


def bench_surrogate(args, vm, gamma, dev, stream):
    """Learned surrogate with fallback: trained on the GPU (HIP forward /
    backward / Adam) on (f, Q) pairs the exact FP32 operator produces from
    (i) states sampled from runs of the lid-driven cavity and (ii) seeded
    near-equilibrium states of a low-Knudsen field, then timed and scored
    against the exact operators on (a) an unseen state of the 4096-point
    cavity and (b) an unseen 4096-point low-Knudsen field."""
    import torch

    from dgfs_hip.solvers.dgfs.scattering import VHSOperator
    from dgfs_hip.surrogate import SpectralSurrogate

    P = args.points
    exact32 = VHSOperator.from_mesh(vm, gamma, 1.0, precision=32, project=True)
    sur = SpectralSurrogate(vm.Nv(), vm.L(), vm.cw(), gamma, 1.0, max_batch=2048, device=dev, seed=0,
                            init_scale=0.3)
    t0 = time.perf_counter()
    xs, lts, ys = [], [], []

    def add(f):
        Q = torch.empty_like(f)
        exact32.eval_contig(f.data_ptr(), Q.data_ptr(), f.shape[0], stream)
        x, lt, y, mo = sur.make_dataset(f, Q)
        keep = mo[:, 5] <= 0.2  # the network only sees points near equilibrium
        xs.append(x[keep]), lts.append(lt[keep]), ys.append(y[keep])
        return int(keep.sum())

    n_cav = 0
    f_cav_eval, cav_step, cav_t = None, 0, 0.0
    if args.sur_cavity_snaps > 0:
        snaps = cavity_snapshots(args, dev, args.sur_cavity_snaps + 1, args.sur_cavity_every,
                                 args.sur_cavity_every)
        for k, (f, step, tc) in enumerate(snaps):
            if k < args.sur_cavity_snaps:
                n_cav += add(f)
                del f
            else:
                f_cav_eval, cav_step, cav_t = f, step, tc  # unseen: one interval after the last
    n_syn = 0
    for c0 in range(0, args.sur_train, 4096):
        nb = min(4096, args.sur_train - c0)
        # near-equilibrium states only: far states go to the exact operator, and
        # their large Q would dominate the mean-square error of the modes
        n_syn += add(near_equilibrium_states(vm, nb, seed=1000 + c0, device=dev, frac_far=0.0))
    x, lt, y = torch.cat(xs), torch.cat(lts), torch.cat(ys)
    torch.cuda.synchronize()
    t_data = time.perf_counter() - t0
    t0 = time.perf_counter()
    losses = sur.train(x, lt, y, epochs=args.sur_epochs, batch=256, lr=1e-3)
    torch.cuda.synchronize()
    t_train = time.perf_counter() - t0
    del x, lt, y, xs, lts, ys
    out = {"unit": "Q(f) evals/s",
           "network": "4 layers, 512 Hermite modes x 32 channels, BF16 weights, FP32 activations, FP32 MFMA",
           "train_states_cavity": n_cav, "train_states_field": n_syn, "train_epochs": args.sur_epochs,
           "train_loss_first_last": [losses[0], losses[-1]], "data_gen_s": t_data, "train_s": t_train}
    have_cavity = f_cav_eval is not None
    if have_cavity:
        res = surrogate_eval(args, vm, sur, exact32, f_cav_eval, dev, stream)
        out.update({"workload": f"lid-driven cavity 16x16 quads p=3 ({f_cav_eval.shape[0]} points), Nv={vm.Nv()}, "
                                f"state after {cav_step} SSP-RK2 steps (t = {cav_t:.4g}), unseen in training",
                    **res})
        del f_cav_eval
    # a harder field: most points off equilibrium by up to 0.3, 5 % far
    f = near_equilibrium_states(vm, P, seed=7, device=dev)
    field = surrogate_eval(args, vm, sur, exact32, f, dev, stream)
    field["workload"] = (f"{P} points of a low-Knudsen field (seeded Maxwellians with Chapman-Enskog "
                         f"perturbations of log-uniform amplitude 1e-3..0.3, 5% bimodal/anisotropic), "
                         f"Nv={vm.Nv()}")
    if have_cavity:
        out["low_knudsen_field"] = field
    else:
        out.update(field)
    del f
    exact32.close()
    sur.close()
    return out


def make_states(vm, npts, seed, device, dtype=None):
    """Seeded bimodal / anisotropic Maxwellians (DGFS convention
    (pi T)^-3/2 exp(-|c-u|^2/T)), renormalised to density 1 on the grid."""
    import numpy as np
    import torch
    rng = np.random.default_rng(seed)
    params = []
    for i in range(npts):
        if i % 2 == 0:
            u = []
            for _ in range(2):
                d = rng.normal(size=3)
                d /= np.linalg.norm(d)
                u.append(d * rng.uniform(0, 1) ** (1 / 3))
            T = rng.uniform(0.5, 2.0, 2)
            params.append((0, np.concatenate([u[0], u[1]]), T))
        else:
            params.append((1, np.zeros(6), rng.uniform(0.3, 3.0, 3)))
    cv = torch.as_tensor(vm.cv(), device=device)
    out = torch.empty((npts, vm.vsize()), dtype=torch.float64, device=device)
    kind = np.array([k for k, _, _ in params])
    U = torch.as_tensor(np.stack([u for _, u, _ in params]), device=device)
    Tb = np.stack([np.resize(T, 3) for _, _, T in params])
    T = torch.as_tensor(Tb, device=device)
    isbi = torch.as_tensor(kind == 0, device=device).view(-1, 1)
    for s0 in range(0, npts, 256):
        s1 = min(npts, s0 + 256)
        u1, u2 = U[s0:s1, 0:3, None], U[s0:s1, 3:6, None]
        t = T[s0:s1, :, None]
        c = cv[None]
        bi = (0.5 * torch.exp(-((c - u1) ** 2).sum(1) / t[:, 0]) / (math.pi * t[:, 0]) ** 1.5
              + 0.5 * torch.exp(-((c - u2) ** 2).sum(1) / t[:, 1]) / (math.pi * t[:, 1]) ** 1.5)
        an = torch.exp(-(c ** 2 / t).sum(1)) / (math.pi ** 1.5 * torch.sqrt(t.prod(1)))
        f = torch.where(isbi[s0:s1], bi, an)
        out[s0:s1] = f / (f.sum(1, keepdim=True) * vm.cw())
    return out


def algorithmic_bytes(nv, K, c):
    """B_Q = 2 c n (3K + 3): one HBM read + write of each of the 3K+3
    transforms of the reference dataflow (complex, c bytes per value)."""
    return 2.0 * c * nv ** 3 * (3 * K + 3)


def own_bytes(nv, K, Nrho, c):
    """Same HBM model priced on this implementation's own transform count:
    K packed inverse transforms, Nrho forward transforms, 3 more."""
    return 2.0 * c * nv ** 3 * (K + Nrho + 3)


def own_flops(nv, K, Nrho):
    """FLOPs of this implementation per eval: K packed complex 3D transforms,
    Nrho forward transforms of S_p, 3 more (prep, finalize), the 3 Nyquist 2D
    transforms per (p,q) and the pointwise products."""
    n = nv ** 3
    t3 = 5.0 * n * math.log2(n)
    t2 = 5.0 * nv * nv * math.log2(nv * nv)
    return (K + Nrho + 3) * t3 + 3 * K * t2 + 24.0 * K * n


def survey_flops(nv, K):
    """F_Q of the reference dataflow: (3K+3) complex 3D transforms of
    5 n log2 n flops plus 24 K n pointwise flops."""
    n = nv ** 3
    return (3 * K + 3) * 5.0 * n * math.log2(n) + 24.0 * K * n


def aosoa_register(f, nupts):
    """The AoSoA distribution register of an element type holding the points
    of f ([point][velocity], point = element * nupts + upt): (nupts, ldim)
    with entry (upt, ((e/32)*vsize + v)*32 + e%32), ldim the row length
    rounded up to 16 doubles (backends/base/types.py AoSoA layout)."""
    import torch
    P, vsize = f.shape
    neles = P // nupts
    nparr = -(-neles // 32) * 32
    ncol = nparr * vsize
    ldim = -(-ncol // 16) * 16
    reg = torch.zeros((nupts, ldim), dtype=f.dtype, device=f.device)
    src = torch.zeros((nparr, nupts, vsize), dtype=f.dtype, device=f.device)
    src[:neles] = f.view(neles, nupts, vsize)
    reg[:, :ncol] = src.view(nparr // 32, 32, nupts, vsize).permute(2, 0, 3, 1).reshape(nupts, ncol)
    return reg, neles, ldim


def from_aosoa(reg, nupts, neles, vsize):
    """Inverse of aosoa_register: [point][velocity]."""
    nparr = -(-neles // 32) * 32
    a = reg[:, :nparr * vsize].reshape(nupts, nparr // 32, vsize, 32).permute(1, 3, 0, 2)
    return a.reshape(nparr, nupts, vsize)[:neles].reshape(neles * nupts, vsize)


def read_traffic(name):
    """HBM bytes per dispatch from the committed FETCH_SIZE / WRITE_SIZE
    counter runs (already scaled by the copy-kernel calibration)."""
    path = os.path.join(ROOT, "profiles", name) if name else ""
    if not name or not os.path.isfile(path):
        return None
    with open(path) as fh:
        return json.load(fh)


def headline(record):
    """The record without its threshold tables and explanatory texts, floats to
    seven digits."""
    def short(x):
        if isinstance(x, dict):
            return {k: short(v) for k, v in x.items() if k not in DETAILS}
        if isinstance(x, list):
            return [short(v) for v in x]
        return float(f"{x:.7g}") if isinstance(x, float) else x

    out = short(record)
    for sec in (out.get("surrogate"), out.get("surrogate", {}).get("low_knudsen_field")):
        if sec:
            keep = ("unit", "workload", "points", "value", "fallback_rate", "rel_l2_vs_fp64", "fallback_threshold",
                    "fallback_threshold_high_modes", "conservation_max_rel", "speedup_vs_fp64", "fastest_within_1e-3",
                    "low_knudsen_field")
            for k in [k for k in sec if k not in keep]:
                del sec[k]
    return out


# explanatory texts of the full record
DETAILS = ("note", "flops_model", "compute_unit", "traffic_source")


def main():
    args = parse()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(json.dumps({"error": "this build runs on one GPU: the collision operator of "
                          "every point is independent and no multi-GPU path is built; "
                          "run with --gpus 1"}))
        sys.exit(2)

    import numpy as np
    import torch

    from dgfs_hip.solvers.dgfs.scattering import VHSOperator
    from dgfs_hip.solvers.dgfs.velocitymesh import DGFSVelocityMesh

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    stream = torch.cuda.current_stream().cuda_stream
    if args.calibrate_copy_mib > 0:
        calibrate_copy(args.calibrate_copy_mib, dev)
    nv, P, K = args.nv, args.points, args.M * args.nrho
    gamma = 2.0 * (1.0 - args.omega)
    vm = DGFSVelocityMesh.from_params(None, nv, args.L, args.nrho, args.M)
    f = make_states(vm, P, seed=0, device=dev)
    Q32 = torch.empty_like(f)
    torch.cuda.synchronize()

    op32 = VHSOperator.from_mesh(vm, gamma, 1.0, precision=32, project=True)
    if args.algorithm:
        op32.set_algorithm(args.algorithm)
    if args.groups:
        op32.set_groups(args.groups)
    # the solver's AoSoA registers of the cavity's element type (16 solution
    # points x 256 elements): the drop-in entry point fs_batch calls
    nupts = args.nupts
    if P % nupts:
        raise SystemExit(f"--points {P} is not a multiple of --nupts {nupts}")
    reg_f, neles, ldim = aosoa_register(f, nupts)
    reg_q = torch.zeros_like(reg_f)

    def step_aosoa():
        op32.eval_aosoa(reg_f.data_ptr(), reg_q.data_ptr(), nupts, ldim, vm.vsize(), neles, 0, neles, stream)

    for _ in range(args.warmup):
        step_aosoa()
    torch.cuda.synchronize()
    op32.set_timing(True)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    e0.record()
    for _ in range(args.steps):
        step_aosoa()
    e1.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ev_ms = e0.elapsed_time(e1)
    tim = op32.get_timing()
    cfg = op32.get_config()
    algo, planar = op32.get_algorithm(), op32.ran_planar()
    op32.set_timing(False)
    ms_per_step = 1e3 * wall / args.steps
    value = P * args.steps / wall
    Q32 = from_aosoa(reg_q, nupts, neles, vm.vsize()).contiguous()
    # the contiguous entry point on the same states
    Qc = torch.empty_like(f)
    op32.eval_contig(f.data_ptr(), Qc.data_ptr(), P, stream)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        op32.eval_contig(f.data_ptr(), Qc.data_ptr(), P, stream)
    torch.cuda.synchronize()
    value_contig = P * args.steps / (time.perf_counter() - t0)
    aosoa_vs_contig = float((Q32 - Qc).abs().max())
    del Qc, reg_q

    gain_ms, gain_n = tim["gain"]
    launch_s = gain_ms / max(gain_n, 1) / 1e3
    pts_per_launch = P * args.steps / max(gain_n, 1)
    # planar-direction gain: per (p, pair of mirrored directions) 3 N lines' worth
    # of moves on each of N planes, N^2 operations a line; the other kernels:
    # their transforms
    flops = args.nrho * (args.M // 2) * 3 * nv ** 4 if planar else own_flops(nv, K, args.nrho)
    achieved_tf = flops * pts_per_launch / launch_s / 1e12
    bq32 = algorithmic_bytes(nv, K, 8)
    traffic, traffic_src = None, None
    tname = {2: f"vhs_gain_rr_fp32_n{nv}_traffic.json", 3: f"vhs_gain_rr_inl_fp32_n{nv}_traffic.json",
             4: f"vhs_gain_rr1_fp32_n{nv}_traffic.json", 5: f"vhs_gain_rr_wl_fp32_n{nv}_traffic.json"}.get(algo, "")
    tr = None if planar else read_traffic(tname)
    if tr and tr.get("points_per_dispatch"):
        traffic = tr["bytes_per_dispatch"] * pts_per_launch / tr["points_per_dispatch"]
        traffic_src = (f"profiles/{tname}: rocprofv3 FETCH_SIZE and WRITE_SIZE runs of this kernel "
                       f"({tr.get('points_per_dispatch')} points per dispatch), scaled by the copy-kernel "
                       f"calibration and to this launch's points; not measured in this run")
    kname = (f"k_vhs_gain_planar<float,{nv}>" if planar
             else f"k_vhs_gain_rr<float,{nv},{'true' if algo == 3 else 'false'}>" if algo in (2, 3)
             else f"k_vhs_gain_rr<float,{nv},false,true>" if algo == 5
             else f"k_vhs_gain_rr1<float,{nv}>" if algo == 4 else f"k_vhs_gain<float,{nv}>")

    line = {
        "metric": METRIC,
        "value": value,
        "unit": "Q(f) evals/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": f"cavity collision batch: {P} points ({nupts} solution points x {neles} elements, "
                        f"AoSoA register), Nv={nv} on [-{args.L:g},{args.L:g}]^3, M={args.M}, "
                        f"Nrho={args.nrho}, omega={args.omega}, FP32 transforms + FP64 invariant projection",
            "entry_point": "dgfs_vhs_eval (AoSoA drop-in, fs_batch)",
            "points": P, "nv": nv, "M": args.M, "Nrho": args.nrho, "omega": args.omega,
            "precision": "fp32+fp64-projection",
            "ngroups": cfg["ngroups"], "persistent_workgroups": cfg["nslots"],
        },
        "value_contiguous_entry_point": value_contig,
        "aosoa_vs_contiguous_max_abs_diff": aosoa_vs_contig,
        "roofline": {
            "bound": "mfma",
            "achieved": achieved_tf,
            "peak": FP32_PEAK / 1e12,
            "unit": "TFLOP/s",
            "frac": achieved_tf * 1e12 / FP32_PEAK,
            "traffic": traffic,
            "traffic_source": traffic_src,
            "kernel": kname,
            "compute_unit": "FP32 matrix cores (the moves) and vector ALU (sums, products, y and z transforms)"
                            if planar else
                            "FP32 vector ALU (FFT butterflies and products; packed FP32 is disabled by the "
                            "build, so 78.6 TFLOP/s of the 157.3 is reachable)",
            "flops_per_eval": flops,
            "flops_model": "the matrix products alone: 3 N^4 per radial node and pair of directions; the "
                           "launch time includes the x-forward pass" if planar else
                           "this kernel's own count: K packed complex 3D transforms, Nrho forward transforms, "
                           "3 more, 3K Nyquist-plane 2D transforms (5 N log2 N each), 24 K n pointwise",
            "points_per_launch": pts_per_launch,
            "avg_launch_ms": launch_s * 1e3,
            "frac_of_unpacked_fp32": achieved_tf * 1e12 / (FP32_PEAK / 2),
            "hbm_counter_gbps": (traffic / launch_s / 1e9) if traffic else None,
            "hbm_counter_frac": (traffic / launch_s / HBM_PEAK) if traffic else None,
            "frac_survey_flops": survey_flops(nv, K) * pts_per_launch / launch_s / FP32_PEAK,
            "frac_ref_dataflow": bq32 * pts_per_launch / launch_s / HBM_PEAK,
            "frac_own_transforms": None if planar else own_bytes(nv, K, args.nrho, 8) * pts_per_launch / launch_s / HBM_PEAK,
            "algorithmic_bytes_per_eval": bq32,
            "note": ("frac = this kernel's FLOPs / FP32 peak (its matrix products and its vector work share the "
                     "SIMDs' issue slots); " if planar else
                     "frac = this kernel's FLOPs / FP32 peak (the kernel keeps every transform on chip and is "
                     "bound by VALU issue, LDS transposes and barriers); ") +
                    "frac_ref_dataflow prices the "
                    "reference dataflow's 3K+3 transforms crossing HBM once (B_Q = 2*8*n*(3K+3)) and "
                    "exceeds 1 because they never do; frac_survey_flops counts the reference dataflow's "
                    "(3K+3) transforms, 2.25x the transform kernels' count",
        },
        "kernel_ms_per_step": {k: v[0] / args.steps for k, v in tim.items()},
        "event_ms_total": ev_ms,
    }

    # plain FP64 path, error of FP32 vs FP64, conservation after projection
    if not args.no_fp64:
        # the plain FP64 drop-in, timed on the same AoSoA register
        op64 = VHSOperator.from_mesh(vm, gamma, 1.0, precision=64, project=False)
        reg_q64 = torch.zeros_like(reg_f)

        def step64():
            op64.eval_aosoa(reg_f.data_ptr(), reg_q64.data_ptr(), nupts, ldim, vm.vsize(), neles, 0, neles,
                            stream)
        step64()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.fp64_steps):
            step64()
        torch.cuda.synchronize()
        w64 = time.perf_counter() - t0
        v64 = P * args.fp64_steps / w64
        alg64, planar64 = op64.get_algorithm(), op64.ran_planar()
        Q64 = from_aosoa(reg_q64, nupts, neles, vm.vsize()).contiguous()
        # the multi-pass FP64 kernel the slab kernel replaced, one timed eval
        # (Q bitwise unused: the default's Q64 is the reference below)
        op64.set_algorithm(1)
        step64()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        step64()
        torch.cuda.synchronize()
        w64mp = time.perf_counter() - t0
        del reg_q64
        # the precision claim compares like with like: FP64 with the same FP64
        # projection (the projection itself moves Q by the spectral method's
        # conservation defect, reported separately)
        op64p = VHSOperator.from_mesh(vm, gamma, 1.0, precision=64, project=True)
        Q64p = torch.empty_like(f)
        op64p.eval_contig(f.data_ptr(), Q64p.data_ptr(), P, stream)
        torch.cuda.synchronize()
        err = float(torch.linalg.norm(Q32 - Q64p) / torch.linalg.norm(Q64p))
        err_unproj = float(torch.linalg.norm(Q32 - Q64) / torch.linalg.norm(Q64))
        proj_size = float(torch.linalg.norm(Q64p - Q64) / torch.linalg.norm(Q64))
        cv = torch.as_tensor(vm.cv(), device=dev)
        phi = torch.stack([torch.ones_like(cv[0]), cv[0], cv[1], cv[2], (cv ** 2).sum(0)])
        inv = (Q32 @ phi.T) * vm.cw()
        absq = Q32.abs().sum(1, keepdim=True) * vm.cw()
        cons = float((inv.abs() / absq).max())
        mom = {}
        for j, name in enumerate(["mass", "momentum_x", "momentum_y", "momentum_z", "energy"]):
            d32 = (Q32 @ phi[j]) * vm.cw()
            d64 = (Q64p @ phi[j]) * vm.cw()
            mom[name] = float((d32 - d64).abs().max() / absq.max())
        line["fp64_plain"] = {"value": v64, "unit": "Q(f) evals/s", "ms_per_step": 1e3 * w64 / args.fp64_steps,
                              "steps": args.fp64_steps, "algorithm": alg64,
                              "kernel": "planar" if planar64 else
                              {6: "slab", 1: "multi-pass"}.get(alg64, str(alg64))}
        line["fp64_multipass"] = {"value": P / w64mp, "unit": "Q(f) evals/s", "ms_per_step": 1e3 * w64mp,
                                  "steps": 1, "note": "the FP64 multi-pass gain kernel (algorithm 1)"}
        line["fp32_vs_fp64_rel_l2"] = err
        line["fp32_vs_fp64_unprojected_rel_l2"] = err_unproj
        line["projection_size_rel_l2"] = proj_size
        line["precision_vs_fp64"] = {
            "fp32_projected_vs_fp64_projected": err,
            "fp32_projected_vs_fp64_plain": err_unproj,
            "projection_size": proj_size,
            "note": "the FP64 projection onto the collision invariants corrects the spectral operator's "
                    "conservation defect, which the reference has too; its size is set by the angular "
                    "design and the velocity box, not by FP32 (tests/test_oracle_vhs.py), so the headline "
                    "FP32 path differs from the plain FP64 path by it and from the projected FP64 path by "
                    "the FP32 rounding alone"}
        line["fp32_speedup_vs_fp64"] = value / v64
        line["conservation_after_projection_max_rel"] = cons
        line["moment_error_vs_fp64_rel"] = mom
        del op64, Q64, op64p, Q64p

    op32.close()
    torch.cuda.empty_cache()
    if args.sur_train > 0:
        line["surrogate"] = bench_surrogate(args, vm, gamma, dev, stream)
        if "fp64_plain" in line:
            v64 = line["fp64_plain"]["value"]
            line["surrogate"]["speedup_vs_fp64"] = line["surrogate"]["value"] / v64
            if "low_knudsen_field" in line["surrogate"]:
                fld = line["surrogate"]["low_knudsen_field"]
                fld["speedup_vs_fp64"] = fld["value"] / v64
            for blk in (line["surrogate"], line["surrogate"].get("low_knudsen_field", {})):
                if blk.get("fastest_within_1e-3"):
                    blk["fastest_within_1e-3"]["speedup_vs_fp64"] = blk["fastest_within_1e-3"]["value"] / v64
                for v in blk.get("sampled_spectral_check", {}).values():
                    v["speedup_vs_fp64"] = v["value"] / v64
        torch.cuda.empty_cache()
    if args.pair_points > 0:
        line["mixed_grid_batch"] = bench_pair(args, dev, stream)
        torch.cuda.empty_cache()
    if args.rhs_steps > 0:
        line["rhs"] = bench_rhs(args, dev)
    if args.vss_points > 0:
        line["vss_mixture"] = bench_vss(args, dev, stream)
        torch.cuda.empty_cache()

    if not args.no_cpu:
        from oracle import vhs as O
        ncores = len(os.sched_getaffinity(0))
        workers = min(ncores, 16)
        ov = O.VelocityMesh(nv, args.L, args.nrho, args.M)
        orc = O.VHSOracle(ov, gamma, 1.0)
        sample = f[: args.cpu_points].cpu().numpy()
        orc.q(sample[:1], workers=workers)
        t0 = time.perf_counter()
        orc.q(sample, workers=workers)
        tc = time.perf_counter() - t0
        t0 = time.perf_counter()
        orc.q(sample[:2], workers=1)
        t1 = time.perf_counter() - t0
        line["cpu_baseline"] = {
            "value": args.cpu_points / tc, "unit": "Q(f) evals/s", "cores": workers,
            "kind": "port",
            "sample": f"FP64 numpy/scipy.fft restatement of the reference dataflow (3K+3 "
                      f"transforms) on the first {args.cpu_points} points of the same workload; "
                      f"1-core rate {2 / t1:.3f} evals/s on 2 points",
            "one_core_value": 2 / t1,
        }

    # every table and note on stderr; the one line on stdout stays short enough
    # to be read whole from the tail of a log
    print("# full record: " + json.dumps(line), file=sys.stderr, flush=True)
    print(json.dumps(headline(line)), flush=True)


if __name__ == "__main__":
    main()
