"""Benchmark: PCG time-to-solution of the POT3D Laplace solve on one MI355X.

Workload (default, --config 5): 301x601x1201 PFCS-style 'open' problem
(214.7 M unknowns), r in [2.5, 10] with a geometric radial mesh, uniform
theta/phi, seeded synthetic Br (16 bipoles + l<=15 background) with the
|Br| treatment and phi=0 at r1, ILU0 preconditioner, stopping at
||b - Ax||2/||b||2 <= 1e-9.  --config 2 runs the 151x301x601 PFSS problem
(r in [1, 2.5], 8 bipoles, phi=0 at 2.5).  A step is one complete solve
with the vectors already resident in HBM.

Reported:
  value        time-to-solution of the reported path, seconds: FP32 inner
               PCG with the FP64 solution (reliable updates), the
               block-Jacobi ILU0 (the reference's per-rank ILU0 on a grid
               cut into 8x16x16 blocks) and the learned warm start (network
               trained on 51x91x181 PCG solutions of the same problem family,
               weights committed under pot3d_amd/weights/, prolonged to the
               fine grid); the network's prediction is inside the timed region
  fp64_plain   the plain FP64 single-rank ILU0 PCG (the drop-in baseline),
               and the speed-up over it; fp64_blockjacobi the FP64 solve with
               the value path's preconditioner (the same-preconditioner
               ratio); mixed the value path without the network
  errors       potential, B field (getb) and magnetic energy of each fast path
               against the FP64 solve, asserted against 1e-8 / 1e-8 / 1e-7
  roofline     the value path's dominant kernel (the FP32 block-Jacobi ILU0
               apply): algorithmic bytes / HIP-event time on the solver's
               stream vs 8 TB/s, and its measured HBM traffic; also the whole
               iteration's algorithmic bytes per iteration time
  cpu_baseline the reference's CPU ifprec=2 algorithm (per-rank diacsr +
               Saad ilu0 + lusol, block-Jacobi over P MPI ranks, P = the host
               cores this job may use) restated in the oracle: a bounded
               sample at this workload, plus a full solve to convergence of
               the 51x91x181 problem of the same family
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
PHI_TOL, B_TOL, E_TOL = 1e-8, 1e-8, 1e-7

from pot3d_amd._hip import Hip  # noqa: E402

# config number -> (problem family, grid, label)
CONFIGS = {
    5: ("open", (301, 601, 1201), "PFCS-style open"),
    2: ("pfss", (151, 301, 601), "PFSS"),
}


def host_cores() -> int:
    """Host cores this job may use: OMP_NUM_THREADS when the environment
    sets it (the GPU host grants a share of its cores), else all."""
    v = os.environ.get("OMP_NUM_THREADS")
    try:
        return max(1, int(v)) if v else (os.cpu_count() or 1)
    except ValueError:
        return os.cpu_count() or 1


def cpu_baseline(workload, family: str, cores: int, sample_iters: int, n_iter_est: int):
    """The reference's CPU ifprec=2 solve on `cores` MPI ranks (the oracle's
    restatement, one OpenMP thread per rank): set-up and `sample_iters`
    iterations timed at this workload and scaled to n_iter_est iterations;
    and the 51x91x181 problem of the same family solved to convergence."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle
    from p3d_driver import workloads
    m = workload.mesh
    topo = oracle.rank_topology(m.nr, m.nt, m.np, cores)
    o = oracle.Oracle(m, workload.pm_r1)
    t0 = time.perf_counter()
    b = o.rhs(workload.br0)
    o.coefs()
    t_coef = time.perf_counter() - t0
    res = o.cgsolve_ranks(b, topo, epscg=1e-9, stop_mode=1, ncgmax=sample_iters)
    per_iter = res["t_iter"] / max(res["ncg"], 1)
    t_ilu = res["t_setup"]
    est = t_coef + t_ilu + per_iter * n_iter_est
    del o, b, res
    # the coarse problem of the same family, to convergence
    wc = workloads.domain_workload(family, workloads.COARSE_GRID, 0)
    mc = wc.mesh
    topc = oracle.rank_topology(mc.nr, mc.nt, mc.np, cores)
    oc = oracle.Oracle(mc, wc.pm_r1)
    t0 = time.perf_counter()
    bc = oc.rhs(wc.br0)
    oc.coefs()
    t_cc = time.perf_counter() - t0
    rc = oc.cgsolve_ranks(bc, topc, epscg=1e-9, stop_mode=1)
    full = {"workload": wc.name, "ranks": list(topc), "ierr": rc["ierr"], "ncg": rc["ncg"],
            "t_total_s": round(t_cc + rc["t_setup"] + rc["t_iter"], 3),
            "t_setup_s": round(t_cc + rc["t_setup"], 3), "t_iter_s": round(rc["t_iter"], 3)}
    return {"value": round(est, 2), "unit": "s (estimated time-to-solution)", "cores": cores,
            "kind": "port", "ranks": list(topo),
            "sample": (f"the oracle's restatement of the reference's CPU ifprec=2 solve "
                       f"(per-rank diacsr + Saad ilu0 + lusol, block-Jacobi over "
                       f"{topo[0]}x{topo[1]}x{topo[2]} ranks, one thread each, stored FP64 "
                       f"operator) on this workload: coefficients {t_coef:.1f} s, ILU0 set-up "
                       f"{t_ilu:.1f} s and "
                       f"{sample_iters} iterations at {per_iter:.3f} s each, scaled to "
                       f"{n_iter_est} iterations (the single-rank ILU0's count: a lower bound, "
                       f"the block-Jacobi cut only adds iterations)"),
            "per_iter_s": round(per_iter, 4), "t_setup_s": round(t_coef + t_ilu, 2),
            "full_solve_coarse": full}


# (name, time_kernel id, algorithmic bytes per unknown, padded-array bytes per point)
KERNELS = [
    # operator 8 + 8 (padded), forward sweep with r -= alpha Ap 32, backward
    # sweep 16, r.z with r.r 16, p update with x 34
    ("pcg_iteration_fp64 (graph replay)", 3, 106, 8),
    ("stencil_fp64 (k_stencil_lds<double>)", 0, 8, 8),
    ("stencil_fp32 (k_stencil_lds<float>)", 1, 4, 4),
    ("ilu_apply_fp64 (k_col_fwd+k_col_bwd<double>)", 2, 32, 0),
    ("ilu_apply_fp32 (column or tile sweeps, float)", 7, 24, 0),
    # r, ap read, r written (runs where the sweeps do not take it)
    ("cg_update_fp64 (k_cg_update<double>)", 4, 24, 0),
    # p, z read, p written, and the solution once per 4 iterations:
    # (4*24 + 16 + 24) / 4
    ("p_update_fp64 (k_p_update_x<double>, x every 4 iterations)", 5, 34, 0),
    ("copy_fp64 (k_copy<double>)", 6, 16, 0),
]


def measure_kernels(s, N: int, padded: int, nr: int, reps: int = 20, graph: bool = True):
    """Average HIP-event time per launch on the solver's stream, algorithmic
    bytes per launch and the achieved bandwidth of each kernel.  graph=False
    leaves out the graph-replayed iteration."""
    table = {}
    for name, kid, per_n, per_pad in KERNELS:
        if kid == 3 and not graph:
            continue
        ms = s.time_kernel(kid, reps if kid not in (2, 7) else 5)
        nbytes = per_n * N + per_pad * padded
        table[name] = {"ms": round(ms, 5), "bytes": nbytes,
                       "GBs": round(nbytes / (ms * 1e-3) / 1e9, 1)}
    return {"table": table}


# Kernels of the value path's iteration: FP32 recurrence with the
# block-Jacobi ILU0 on register tiles.  (name, time_kernel id, algorithmic
# bytes per unknown, padded-array bytes per point).  From 2^26 unknowns the
# library folds the residual update into the ILU's forward sweep
# (P3D_OPT_FUSE_RESIDUAL = -1): one kernel sequence or the other.
FUSE_RESIDUAL_MIN_N = 1 << 26
VALUE_KERNELS_FUSED = [
    # r, ap, dinv read, r, y written (forward); y, dinv read, z written
    ("ilu_apply_fp32_blockjacobi_with_r_update (k_tile_fwd_reg<float, 16, false, true>"
     "+k_tile_bwd_reg<float>)", 11, 32, 0),
]
VALUE_KERNELS_SEPARATE = [
    # below 2^26 unknowns a workgroup per block marches the block's diagonals
    ("ilu_apply_fp32_blockjacobi (k_tile_fwd_blk+k_tile_bwd_blk<float>, block-persistent)",
     7, 24, 0),
    # r, ap read, r written (tile-major)
    ("r_update_fp32 (k_r_update)", 9, 12, 0),
]
VALUE_KERNELS_REST = [
    ("stencil_fp32 (k_stencil_lds<float>)", 1, 4, 4),
    # per iteration of a group of 4: p, z (tile-major, gathered) read, p
    # written (12 B) on every iteration, and on the group's last one also
    # the FP64 solution read and written (16) and the group's 3 earlier
    # directions read (12): (4*12 + 28) / 4 = 19 B
    ("p_update_fp32_fp64x (k_p_update_x<float>, x every 4 iterations)", 8, 19, 0),
    # r, z read: r.z and r.r
    ("rz_rr_dot_fp32 (k_dot2<float>, tile order)", 10, 8, 0),
]


def value_kernels(N: int):
    """The value path's kernel sequence at N unknowns (its ILU apply first)."""
    head = VALUE_KERNELS_FUSED if N >= FUSE_RESIDUAL_MIN_N else VALUE_KERNELS_SEPARATE
    return head + VALUE_KERNELS_REST


def set_fast_ilu(s, args):
    """The block-Jacobi ILU0 of the fast paths (the reference's per-rank
    ILU0 on a grid decomposed into that many blocks)."""
    from pot3d_amd import _lib
    blocks = tuple(int(v) for v in args.blocks.split(","))
    for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T, _lib.OPT_ILU_BLOCKS_P),
                      blocks):
        s.set_option(key, v)
    s.set_option(_lib.OPT_TILE_K, args.tile_k)
    s.set_option(_lib.OPT_TILE_STAGE, args.tile_stage)
    return blocks


def measure_value_kernels(s, N: int, padded: int, nr: int, reps: int = 5):
    """The value path's kernels (set_fast_ilu applied), timed as
    measure_kernels; the ILU apply is the dominant one, so it is the
    roofline kernel.  Also the algorithmic bytes of one iteration."""
    table = {}
    kernels = value_kernels(N)
    for name, kid, per_n, per_pad in kernels:
        ms = s.time_kernel(kid, reps)
        nbytes = per_n * N + per_pad * padded
        table[name] = {"ms": round(ms, 5), "bytes": nbytes,
                       "GBs": round(nbytes / (ms * 1e-3) / 1e9, 1)}
    name = kernels[0][0]
    iter_bytes = sum(v["bytes"] for v in table.values())
    iter_ms = sum(v["ms"] for v in table.values())
    return {"table": table, "dominant": dict(name=name, **table[name]),
            "iter_bytes": iter_bytes, "kernels_ms": iter_ms}


def measured_traffic(grid: str, kernel: str):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 PMC
    summary (FETCH_SIZE + WRITE_SIZE, calibrated on a plain copy) for this
    grid, or None when there is none."""
    path = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        with open(path) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    k = t.get(grid, {}).get(kernel)
    return None if k is None else int(k["fetch_bytes"] + k["write_bytes"])


def default_weights(family: str) -> str:
    return os.path.join(ROOT, "pot3d_amd", "weights", f"warmstart_{family}_51x91x181.npz")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3, help="timed solves of the value path")
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--ref-runs", type=int, default=1,
                    help="timed solves of each comparison path (FP64 plain, FP64 "
                         "block-Jacobi, mixed without the network)")
    ap.add_argument("--config", type=int, default=5, choices=sorted(CONFIGS))
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-iters", type=int, default=3,
                    help="iterations of the CPU sample at the full workload")
    ap.add_argument("--kernels-only", action="store_true",
                    help="only time the kernels (for profiler runs)")
    ap.add_argument("--profile-solve", action="store_true",
                    help="one value-path solve without graph capture (for kernel traces)")
    ap.add_argument("--mixed-mode", type=int, default=2,
                    help="1 restarted defect correction, 2 reliable updates")
    ap.add_argument("--weights", type=str, default="",
                    help="warm-start weights (.npz from pot3d_amd.train_warmstart); default "
                         "the committed ones of the problem family; 'none' skips the network")
    ap.add_argument("--blocks", type=str, default="8,16,16",
                    help="block-Jacobi ILU0 blocks (r,theta,phi) of the fast paths; "
                         "1,1,1 = single-rank ILU0")
    ap.add_argument("--tile-k", type=int, default=16,
                    help="planes per ILU tile of the block-Jacobi fast paths (16, 32, 64)")
    ap.add_argument("--tile-stage", type=int, default=2,
                    help="ILU tiles of the fast paths held in registers (2), staged in LDS "
                         "by the marching wave alone (1) or by planes/8 waves (0)")
    ap.add_argument("--levels", action="store_true",
                    help="also time the FP64 solve with hyperplane-level trisolves")
    ap.add_argument("--guess-check", type=int, default=2,
                    help="1 residual rule, 2 A-norm rule for accepting the learned guess")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: the library has no multi-GPU path "
              f"(--gpus {args.gpus} requested); run with --gpus 1.", file=sys.stderr)
        sys.exit(2)

    from p3d_driver import workloads
    family, grid, label = CONFIGS[args.config]
    gname = "x".join(map(str, grid))
    t0 = time.perf_counter()
    w = workloads.config(args.config)
    dom = workloads.DOMAINS[family]
    print(f"[bench] workload {w.name} N={w.N} built in {time.perf_counter() - t0:.1f}s",
          file=sys.stderr, flush=True)
    wpath = args.weights or default_weights(family)
    use_net = wpath != "none" and not args.kernels_only
    if use_net and not os.path.exists(wpath):
        print(f"[bench] no warm-start weights at {wpath}: value path without the network",
              file=sys.stderr, flush=True)
        use_net = False
    wc = workloads.domain_workload(family, workloads.COARSE_GRID, 0) if use_net else None
    cores = host_cores()

    from pot3d_amd import _lib, solver
    hip = Hip()
    N = w.N
    nr, nt, np_ = grid
    s = solver.Pot3dSolver(w.mesh, w.pm_r1, 2)
    s.set_br0(w.br0)
    s.set_option(_lib.OPT_STOP, 1)
    rhs = s.rhs()
    if args.kernels_only:
        kern = measure_kernels(s, N, nr * nt * np_, nr, reps=5, graph=False)
        set_fast_ilu(s, args)
        vkern = measure_value_kernels(s, N, nr * nt * np_, nr)
        print(json.dumps({"workload": w.name, "unknowns": N, "kernels": kern["table"],
                          "value_path_kernels": vkern["table"]}))
        s.close()
        return
    d_x = hip.malloc(8 * N)
    d_b = hip.malloc(8 * N)
    zero = np.zeros(N)

    def run(mixed: int, guess=None):
        """One timed solve; guess(d_x) writes the initial guess on the device
        inside the timed region (None: the zero guess, copied before)."""
        s.set_option(_lib.OPT_MIXED, mixed)
        s.set_option(_lib.OPT_GUESS_CHECK, args.guess_check if guess else 0)
        hip.h2d(d_x, zero)
        hip.h2d(d_b, rhs)
        hip.sync()
        t = time.perf_counter()
        if guess:
            guess(d_x)
        ierr, ncg, epsn = s.solve_dev(d_x, d_b, 1e-9, ncgmax=20000)
        hip.sync()
        dt = time.perf_counter() - t
        st = s.stats()
        assert ierr == 0, f"solve did not converge ({st})"
        return dt, st

    def timed(label, mixed, guess=None, warmup=0, steps=1):
        for _ in range(warmup):
            run(mixed, guess)
        ts = []
        for _ in range(steps):
            dt, st = run(mixed, guess)
            ts.append(dt)
            print(f"[bench] {label}: {dt:.3f}s ncg={st['ncg']} outer={st['n_outer']} "
                  f"guess={st['guess']} relres={st['true_relres']:.2e}", file=sys.stderr,
                  flush=True)
        x = np.empty(N)
        hip.d2h(x, d_x)
        return ts, st, x

    if args.profile_solve:
        # one value-path solve with every kernel launched on its own
        set_fast_ilu(s, args)
        s.set_option(_lib.OPT_GRAPH, 0)
        ts, st, _ = timed("mixed block-Jacobi ILU0 PCG, no graph", args.mixed_mode)
        print(json.dumps({"workload": w.name, "profile_solve_s": round(ts[0], 4),
                          "ncg": st["ncg"]}))
        s.close()
        return

    # FP64 plain ILU0 PCG (drop-in baseline: the single-rank ILU0)
    t64, st64, x64 = timed("fp64 ILU0 PCG", 0, steps=args.ref_runs)
    phi64 = s.fill_phi(x64)
    B64 = s.getb(phi64)
    w64 = s.magnetic_energy(phi64)
    del phi64
    tlv = None
    if args.levels:
        s.set_option(_lib.OPT_SWEEP, 1)
        dt, stlv = run(0)
        tlv = (dt, stlv["ncg"])
        print(f"[bench] fp64 ILU0 PCG, hyperplane-level trisolves: {dt:.3f}s ncg={stlv['ncg']}",
              file=sys.stderr, flush=True)
        s.set_option(_lib.OPT_SWEEP, 0)
    kern = measure_kernels(s, N, nr * nt * np_, nr)
    blocks = set_fast_ilu(s, args)
    vkern = measure_value_kernels(s, N, nr * nt * np_, nr)
    tbj, stbj, _ = timed(f"fp64 block-Jacobi{blocks} ILU0 PCG", 0, steps=args.ref_runs)

    def errs(x):
        """phi, B and energy of x against the FP64 solve (max relative to the
        largest magnitude; energy per component), asserted on the bars."""
        phi = s.fill_phi(x)
        dphi = float(np.max(np.abs(x - x64)) / np.max(np.abs(x64)))
        B = s.getb(phi)
        dB = max(float(np.max(np.abs(g - r)) / np.max(np.abs(r))) for g, r in zip(B, B64))
        wx = s.magnetic_energy(phi)
        dE = float(np.max(np.abs(wx - w64) / np.abs(w64)))
        assert dphi <= PHI_TOL and dB <= B_TOL and dE <= E_TOL, (dphi, dB, dE)
        return {"max_rel_dphi": dphi, "max_rel_dB": dB, "max_rel_denergy": dE}

    # mixed precision from the zero guess
    steps_mx = args.ref_runs if use_net else args.steps
    tmx, stmx, xmx = timed(f"mixed(mode {args.mixed_mode}) block-Jacobi ILU0 PCG",
                           args.mixed_mode, warmup=0 if use_net else args.warmup, steps=steps_mx)
    err_mx = errs(xmx)
    del xmx
    tbest, stbest, vlabel, err_best = tmx, stmx, "mixed", err_mx
    result_ws = None
    if use_net:
        from pot3d_amd import warmstart as W
        net, meta = W.WarmStartNet.load(wpath, wc.mesh, wc.pm_r1)
        sc = solver.Pot3dSolver(wc.mesh, wc.pm_r1, 2)
        # the fine problem's Br map (seed 0) on the coarse mesh
        brc = wc.br0
        sc.set_br0(brc)
        tab = W.prolong_tables(wc.mesh, w.mesh)
        d_phic = hip.malloc(8 * wc.mesh.nr * wc.mesh.nt * wc.mesh.np)

        def guess(dx):
            xc = net.predict(brc)
            phic = sc.fill_phi(xc)
            hip.h2d(d_phic, phic)
            W.prolong_dev_noalloc(tab, d_phic, dx)

        twl, stwl, xwl = timed(f"mixed(mode {args.mixed_mode}) + learned block-Jacobi ILU0 PCG",
                               args.mixed_mode, guess, warmup=args.warmup, steps=args.steps)
        err_wl = errs(xwl)
        del xwl
        # quality of the guess alone
        hip.h2d(d_x, zero)
        guess(d_x)
        xg = np.empty(N)
        hip.d2h(xg, d_x)
        g_err = float(np.linalg.norm(xg - x64) / np.linalg.norm(x64))
        g_res = float(np.linalg.norm(rhs - s.ax(xg)) / np.linalg.norm(rhs))
        del xg
        result_ws = {
            "weights": os.path.relpath(wpath, ROOT), "coarse_grid": "51x91x181",
            "pairs": int(meta.get("pairs", 0)), "epochs": float(meta.get("epochs", 0)),
            "val_guess_rel_err_coarse": float(meta.get("val_guess_rel_err", float("nan"))),
            "params": net.nparams, "guess_rel_err": g_err, "guess_relres": g_res,
            "guess_check_mode": args.guess_check, "guess_kept": stwl["guess"] == 1,
            "mixed_learned_s": round(min(twl), 4), "mixed_learned_ncg": stwl["ncg"],
            "iterations_saved_frac": round(1.0 - stwl["ncg"] / stmx["ncg"], 4),
            "errors_vs_fp64": err_wl}
        if min(twl) < min(tbest):
            tbest, stbest, vlabel, err_best = twl, stwl, "mixed+learned", err_wl
        net.close()
        sc.close()
        hip.free(d_phic)

    dk = vkern["dominant"]
    roof = {"kernel": dk["name"], "bound": "hbm", "achieved": dk["GBs"], "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": round(dk["GBs"] / HBM_PEAK_GBS, 4),
            "traffic": measured_traffic(gname, dk["name"]),
            "avg_ms": dk["ms"], "bytes_per_launch": dk["bytes"]}
    best = min(tbest)
    ms_iter = 1e3 * best / max(stbest["ncg"], 1)
    iter_roof = {"bytes_per_iteration": vkern["iter_bytes"], "ms_per_iteration": round(ms_iter, 4),
                 "achieved": round(vkern["iter_bytes"] / (ms_iter * 1e-3) / 1e9, 1),
                 "frac": round(vkern["iter_bytes"] / (ms_iter * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                 "kernels_ms_sum": round(vkern["kernels_ms"], 4)}
    st_name = "stencil_fp64 (k_stencil_lds<double>)"
    per_iter64 = min(t64) / max(st64["ncg"], 1)
    out = {
        "metric": "PCG time-to-||r||/||b||<=1e-9 (s): mixed+learned vs FP64 plain; "
                  "stencil HBM GB/s",
        "value": round(best, 4), "unit": "s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(1e3 * float(np.mean(tbest)), 2),
        "higher_is_better": False, "scaling": "strong", "vs_baseline": None,
        "dtype": "f64 outer / f32 inner", "data": "synthetic (seeded bipole+harmonic Br)",
        "config": {"workload": f"{label} {gname}, r in [{dom['r0']}, "
                               f"{dom['r1']}], {dom['n_bipoles']} bipoles, option "
                               f"'{dom['option']}', ILU0 PCG to ||r||2/||b||2<=1e-9",
                   "unknowns": N, "precond": "ILU0 (D-ILU); fast paths block-Jacobi ILU0",
                   "epscg": 1e-9, "value_path": vlabel, "mixed_mode": args.mixed_mode},
        "fp64_plain_s": round(min(t64), 4), "fp64_plain_ncg": st64["ncg"],
        "fp64_blockjacobi_s": round(min(tbj), 4), "fp64_blockjacobi_ncg": stbj["ncg"],
        "mixed_s": round(min(tmx), 4), "mixed_ncg": stmx["ncg"], "mixed_outer": stmx["n_outer"],
        "value_ncg": stbest["ncg"],
        "speedup_vs_fp64": round(min(t64) / best, 3),
        "speedup_same_precond": round(min(tbj) / best, 3),
        "speedup_precision_only": round(min(tbj) / min(tmx), 3),
        "ilu_blocks": list(blocks), "ilu_tile_k": args.tile_k,
        "ilu_tile_stage": args.tile_stage,
        "fp64_levels_s": None if tlv is None else round(tlv[0], 4),
        "fp64_levels_ncg": None if tlv is None else tlv[1],
        "errors_vs_fp64": {"bars": [PHI_TOL, B_TOL, E_TOL], "mixed": err_mx,
                           "value_path": err_best},
        "learned": result_ws,
        "fp64_ms_per_iter": round(1e3 * per_iter64, 4),
        "stencil_fp64_GBs": kern["table"][st_name]["GBs"],
        "kernels": kern["table"],
        "value_path_kernels": vkern["table"],
        "roofline": roof, "iteration_roofline": iter_roof,
    }
    s.close()
    hip.free(d_x)
    hip.free(d_b)
    del x64, B64, rhs
    cpu = None
    if not args.no_cpu:
        print(f"[bench] CPU baseline on {cores} cores", file=sys.stderr, flush=True)
        try:
            cpu = cpu_baseline(w, family, cores, args.cpu_iters, st64["ncg"])
        except Exception as e:  # reported, not fatal
            cpu = {"error": repr(e)}
    out["cpu_baseline"] = cpu
    print(json.dumps(out))


if __name__ == "__main__":
    main()
