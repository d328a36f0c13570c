"""Benchmark: time per Newton step to FP64 residual 1e-8 on the 2M-triangle meandering
channel (one MI355X).

The deck's floodplains rise away from the main channel, so that their outer parts lie above
the initial water level: drying and rewetting (method 2, on the device) takes them out of
the system before the first Newton step, as the flow cycle's call at its first step does
(the set-up of the wet model after that call is reported, not timed).
One step = one Newton step of the UVS2D system from the deck's initial state (the state is
uploaded again before every step, outside the timed region, so every step solves the same
system): the drying and rewetting call (no element changes: the device pass and the flags'
download), nodal friction and inlet set-up, FP64 assembly, L2 scaling, FP32 copy of the
matrix, ILU(0) factorisation, coarse-space factorisation, the Krylov solve in FP32 inside
FP64 iterative refinement to ||b - J x|| / ||b|| <= 1e-8 (FP64 J), Newton update.  The
inputs (mesh, pattern, schedules) are resident on the device before the timed region.

Printed (one JSON line):
* value: the step time of the FP32/FP64 path (FGMRES(15) with the two-level
  preconditioner: coarse correction + strip ILU(0) sweeps), Newton steps/s and Krylov
  GDOF-iterations/s (equations x iterations / solve time);
* kernels: every kernel class's launches, time per step and share of it, algorithmic bytes
  per launch and fraction of the HBM peak, from HIP events on the library's stream over the
  timed steps; roofline: the class with the largest share;
* comparison: an 80-cross-section reach of the same generator on which the plain FP64
  ILU0-BiCGStab path reaches 1e-8 within a benchmark run, both paths timed to a true FP64
  residual of 1e-8, and the reference program's own CPU step on the same reach;
* plain_fp64_2M: the plain path on the 2M system run for a bounded number of iterations
  (its time to 1e-8 there exceeds a benchmark run; elapsed / value bounds the speedup);
* learned: the same Newton step with the learned network correcting the two-level
  preconditioner (weights rismo2d_amd/mpnn_meander.npy, trained by
  `python -m rismo2d_amd.mpnn` on 200k-element reaches of other seeds), or null with the
  reason;
* cpu_baseline: the reference program (built from its sources) on the comparison reach, one
  core, with its DOF-iterations/s beside the GPU paths' on the same reach.

    python bench.py [--steps K] [--warmup W] [--gpus 1]
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

METRIC = "time to FP64 residual 1e-8 per Newton step: learned+FP32 vs plain FP64"
HBM_PEAK = 8.0e12          # MI355X HBM3E, bytes/s
CROSS = 320                # cross-sections' cells of the meander generator


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--n-along", type=int, default=3200)
    ap.add_argument("--n-across", type=int, default=CROSS)
    ap.add_argument("--strips", type=int, default=0)
    ap.add_argument("--segments", type=int, default=0, help="segments per strip (0: blocks of about 560 rows)")
    ap.add_argument("--coarse", type=int, default=-1,
                    help="coarse segments per strip (-1: automatic, 0: none)")
    ap.add_argument("--max-iter", type=int, default=1000, help="Krylov iterations per refinement sweep")
    ap.add_argument("--mkyrl", type=int, default=15, help="FGMRES restart length")
    ap.add_argument("--eps", type=float, default=1e-2, help="inner relative tolerance per sweep")
    ap.add_argument("--refine-max", type=int, default=8)
    ap.add_argument("--plain-iters", type=int, default=10,
                    help="BiCGStab iterations of the bounded plain FP64 run on the 2M system")
    ap.add_argument("--plain-rise", type=float, default=0.012,
                    help="floodplain rise (m/m) away from the main channel; > 0: the outer "
                         "floodplains are dry and drying and rewetting is active")
    ap.add_argument("--cmp-along", type=int, default=80,
                    help="cross-sections of the comparison reach (0: no comparison)")
    ap.add_argument("--learned", default=os.path.join(HERE, "rismo2d_amd", "mpnn_meander.npy"),
                    help="weights of the learned preconditioner (numpy float32); the learned "
                         "leg runs when the file exists")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--kernels-only", action="store_true",
                    help="profiling run: build and factor the system, time the FP32 SpMV and "
                         "strip sweeps, run a plain device copy of known size, print their "
                         "times and exit (no Newton step, no JSON benchmark line)")
    return ap.parse_args()


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def reach_deck(n_along, plain_rise, n_across=CROSS):
    """A reach of the benchmark's meander generator at the benchmark's resolution."""
    from rismo2d_amd import deck as dk
    return dk.meander(n_along=n_along, n_across=n_across, reach=10000.0 * n_along / 3200,
                      plain_rise=plain_rise)


def dry_setup(c, rise):
    """The flow cycle's first drying and rewetting call and the set-up of the wet model it
    causes; returns its record (None without a floodplain rise)."""
    if rise <= 0.0:
        return None
    n_all = c.n
    t0 = time.perf_counter()
    dried, wetted = c.dry_rewet()
    t = time.perf_counter() - t0
    _, ef = c.wetdry()
    rec = {"plain_rise": rise, "dried_elements": int(dried), "wetted_elements": int(wetted),
           "dry_elements": int((ef == 1).sum()), "marsh_elements": int((ef == 2).sum()),
           "equations_all_wet": n_all, "equations": c.n, "first_call_and_set_up_s": t}
    log(f"drying: {dried} elements dry, {rec['marsh_elements']} marsh, {n_all} -> {c.n} "
        f"equations; call and set-up of the wet model {t:.2f}s")
    return rec


def cpu_baseline(na, rise):
    """The reference program itself when its build (oracle/_ref/rismo_harness, compiled from
    the reference's sources) is present, else the oracle; both on one core, on the
    comparison reach."""
    exe = os.path.join(HERE, "oracle", "_ref", "rismo_harness")
    if os.path.exists(exe):
        try:
            return cpu_baseline_reference(exe, na, rise)
        except Exception as e:      # noqa: BLE001 - a failed baseline falls back, never stops
            log(f"reference baseline failed ({e}); timing the oracle instead")
    return cpu_baseline_port(na, rise)


def _cpu_seconds(field):
    """'h:mm:ss:cc' of the reference's report (REPORT::PrintTime) in seconds."""
    h, m, sec, cc = (int(v) for v in field.split(":"))
    return 3600 * h + 60 * m + sec + cc / 100.0


CPU_ITERS = 400            # BiCGStab iterations of the bounded CPU sample


def cpu_baseline_reference(exe, na, rise):
    """One Newton step of the reference program on the comparison reach: its own drying
    and rewetting at the step's start (with a floodplain rise) and set-up of the wet model,
    numbering, assembly, ILU(0) and BiCGStab to 1e-8 bounded at CPU_ITERS iterations (its
    FP32-stored matrix stalls above 1e-8 on the dried reach), written as its input files;
    the value is the CPU time its report gives for the time step (the report's last CPU
    line), with the iterations run and the accuracy reached."""
    import re
    import subprocess
    import tempfile
    from rismo2d_amd import deck as dk
    d = reach_deck(na, rise)
    # drying frequency 0: the flow cycle of one Newton step calls it before that step
    # (EqsUVS2D.cpp:201-206); 1000: never
    dry = "2 0 0.001 0.005 100 5" if rise > 0 else "2 1000 0.001 0.005 100 5"
    with tempfile.TemporaryDirectory() as wd:
        dk.write_reference_deck(d, wd, solver=f"1 6 1 0 60 {CPU_ITERS} 1.0e-8", maxiter=1,
                                dryrew=dry)
        subprocess.run([exe, "input.dat"], cwd=wd, check=True, timeout=300,
                       stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        rep = open(os.path.join(wd, "report.txt")).read()
    cpu = re.findall(r"\bCPU:\s+(\d+:\d+:\d+:\d+)", rep)
    it = re.findall(r"P_BCGSTABD::Iterate\)\s+(\d+)\. Iteration \| accuracy = (\S+)", rep)
    neq = re.findall(r"number of equations\D*(\d+)", rep)
    if not cpu or not it:
        raise RuntimeError("no timing or iteration record in the reference's report")
    its, acc = int(it[-1][0]), float(it[-1][1])
    return dict(value=_cpu_seconds(cpu[-1]), unit="s per Newton step", cores=1,
                kind="reference", iters=its, accuracy=acc,
                sample=(f"meander {na}x{CROSS} reach of the benchmark's generator "
                        f"({d.n_elems} triangles" +
                        (f", floodplains rising {rise:g} m/m" if rise > 0 else "") +
                        "), one Newton step of the reference program built from its sources: " +
                        ("drying and rewetting and the wet model's set-up, " if rise > 0 else "") +
                        f"numbering, assembly, ILU(0), BiCGStab {its} it (bounded at "
                        f"{CPU_ITERS}) to accuracy {acc:.1e}; CPU time of the step from its "
                        "report, 1 core (the reference is single-threaded)"))


def cpu_baseline_port(na, rise):
    """The oracle (C restatement of the reference's path, one core) on the comparison
    reach: one Newton step, drying and rewetting (with a floodplain rise), FP64 assembly +
    ILU(0) + BiCGStab to 1e-8."""
    from oracle import pyoracle as po
    d = reach_deck(na, rise)
    m = po.OracleModel(d)
    m.set_params()
    t0 = time.perf_counter()
    if rise > 0:
        m.dry_rewet()
    m.prepare()
    rp, cols = m.pattern()
    A, B = m.assemble(64)
    po.scale(rp, A, B)
    L, _ = po.ilu0_factor(rp, cols, A)
    X, conv, its, acc = po.bicgstab(rp, cols, A, L, B, max_iter=CPU_ITERS, eps=1e-8)
    t = time.perf_counter() - t0
    return dict(value=t, unit="s per Newton step", cores=1, kind="port", iters=its, accuracy=acc,
                sample=(f"meander {na}x{CROSS} reach of the benchmark's generator "
                        f"({d.n_elems} triangles), one Newton step with the oracle: FP64 "
                        f"assembly, ILU(0), BiCGStab {its} it (bounded at {CPU_ITERS}) to "
                        f"{acc:.1e}, 1 core"))


def kernels_only(c, n, a):
    """The system of the first Newton step (FP64 assembly, L2 scaling, FP32 copy), its strip
    ILU(0) and coarse space in FP32, six timed FP32 SpMVs and five applications of the
    two-level preconditioner (its block sweeps with the coarse prolongation folded, as in the
    Newton step), then three plain copies of an n-vector (the identity preconditioner's
    device copy: 8n bytes read, 8n written), the reference size for calibrating HBM byte
    counters."""
    from rismo2d_amd import rmx as R
    c.assemble(R.F64)
    c.scale_l2()
    c.convert(R.F32)
    c.silu0_factor(R.F32)
    c.coarse_factor(R.F32)
    x = np.random.default_rng(0).standard_normal(n)
    c.spmv(x, R.F32)                          # brings the row-group values up to date
    c.kernel_stats(True)
    for _ in range(6):
        c.spmv(x, R.F32)
    for _ in range(5):
        c.precond_apply(R.PREC_SILU0C, x, R.F32)
    ks = c.kernel_stats(False)
    for _ in range(3):
        c.precond_apply(R.PREC_NONE, x, R.F32)
    rec = {"n": n, "nnz": c.nnz, "copy_bytes_each_way": 8 * n}
    for name in ("spmv", "sweeps_block", "sweep_lower", "sweep_upper"):
        sec, byt, cnt = ks[name]
        if cnt:
            rec[name] = {"launches": cnt, "avg_ms": sec / cnt * 1e3, "bytes": byt / cnt}
    print(json.dumps(rec), flush=True)
    c.close()


def fast_opts(a, R, refine_tol=1e-8):
    pk = R.PREC_SILU0C if a.coarse != 0 else R.PREC_SILU0
    return dict(method=R.FGMRES, prec=R.F32, precond=pk, max_iter=a.max_iter, mkyrl=a.mkyrl,
                eps=a.eps, refine=True, refine_tol=refine_tol, refine_max=a.refine_max)


# plain FP64 path: reference-order ILU(0), BiCGStab, FP64 refinement until the true FP64
# residual is 1e-8 (each sweep solves to the remaining factor)
def plain_opts(R, max_iter):
    return dict(method=R.BICGSTAB, prec=R.F64, precond=R.PREC_ILU0, max_iter=max_iter, eps=1e-8,
                refine=True, refine_tol=1e-8, refine_max=4)


def comparison(R, a):
    """Both paths on the comparison reach, each timed over one Newton step from the initial
    state to a true FP64 residual of 1e-8 (the step's factorisations included)."""
    d = reach_deck(a.cmp_along, a.plain_rise)
    c = R.Context(0)
    c.upload_mesh(d)
    c.set_params()
    c.set_coarse(a.coarse)
    c.set_strips(a.strips, a.segments)
    c.prepare()
    wd = dry_setup(c, a.plain_rise)
    n = c.n
    out = {"workload": f"meander {a.cmp_along}x{CROSS} reach of the same generator, "
                       f"{d.n_elems} triangles, {n} equations, {c.nnz} nnz",
           "drying": wd}
    for name, opts in (("fast", fast_opts(a, R)), ("plain_fp64", plain_opts(R, 6000))):
        c.state_upload(d.U0, d.V0, d.S0)
        if wd:
            c.dry_rewet()
        c.newton_step(**opts)                    # warm-up (schedules, first-touch)
        c.state_upload(d.U0, d.V0, d.S0)
        t0 = time.perf_counter()
        if wd:
            assert c.dry_rewet() == (0, 0)
        st = c.newton_step(**opts)
        t = time.perf_counter() - t0
        its = max(st.solve.iters, 1)
        out[name] = {"s_per_newton_step": t, "converged": bool(st.solve.converged),
                     "true_resid": st.solve.true_resid, "krylov_iters": st.solve.iters,
                     "factor_s": st.t_factor, "solve_s": st.t_solve,
                     "dof_iters_per_s": n * its / st.t_solve}
        log(f"comparison {name}: {t:.2f} s per step ({st.solve.iters} it, residual "
            f"{st.solve.true_resid:.1e}, factor {st.t_factor:.2f} s)")
    out["speedup_fast_vs_plain"] = out["plain_fp64"]["s_per_newton_step"] / out["fast"]["s_per_newton_step"]
    out["n_eq"] = n
    c.close()
    return out


KERNEL_NAMES = {"ilu_factor": "k_unit_flow (dataflow ILU(0) factorisation by nodes, FP32)",
                "sweep_lower": "k_sweep_stage lower (strip ILU(0))",
                "sweep_upper": "k_sweep_stage upper (strip ILU(0) + coarse prolongation)",
                "spmv": "k_spmv_grp (FP32 row-group SpMV)",
                "coarse": "coarse correction (restrict, block cyclic reduction, A P residual)",
                "gram_schmidt": "k_gs_dots + k_gs_update (FP32 basis)",
                "resid_fp64": "k_spmv<double> (FP64 refinement residual)",
                "sweeps_block": "k_block_sweep, up to 3,584 blocks k_chunk_sweep (strip ILU(0), both triangles, "
                                "+ coarse prolongation)"}
TRAFFIC_KEYS = {"sweep_lower": "silu_sweep_fwd", "sweep_upper": "silu_sweep_bwd", "spmv": "spmv_f32",
                "sweeps_block": "silu_block_sweep"}


def main():
    a = parse()
    if a.gpus != 1:
        print(f"bench.py runs on one GPU; --gpus {a.gpus} is not supported (the multi-GPU "
              "path is not built)", file=sys.stderr)
        sys.exit(2)
    from rismo2d_amd import deck as dk

    # the CPU baseline first: it starts the reference program as a child process, which is
    # done before this process loads the HIP library or touches the GPU
    cpu = None
    if not a.no_cpu and not a.kernels_only and a.cmp_along > 0:
        try:
            cpu = cpu_baseline(a.cmp_along, a.plain_rise)
            log(f"cpu baseline: {cpu['value']:.1f}s ({cpu['sample']})")
        except Exception as e:       # the oracle library is test infrastructure: report its absence
            log(f"cpu baseline unavailable: {e}")

    from rismo2d_amd import rmx as R

    t = time.perf_counter()
    d = dk.meander(n_along=a.n_along, n_across=a.n_across, reach=10000.0 * a.n_along / 3200,
                   plain_rise=a.plain_rise)
    log(f"deck {a.n_along}x{a.n_across}: {d.n_elems} triangles, {d.n_nodes} nodes "
        f"({time.perf_counter() - t:.1f}s)")
    c = R.Context(0)
    c.upload_mesh(d)
    c.set_params()
    c.set_coarse(a.coarse)
    c.set_strips(a.strips, a.segments)
    t = time.perf_counter()
    n = c.prepare()
    log(f"prepare: {n} equations, {c.nnz} non-zeros ({time.perf_counter() - t:.1f}s)")
    wet = dry_setup(c, a.plain_rise)
    n = c.n

    if a.kernels_only:
        kernels_only(c, n, a)
        return
    opts = fast_opts(a, R)

    def reset():
        # the deck's initial state again (host upload, outside the timed region), so that
        # every step solves the same system
        c.state_upload(d.U0, d.V0, d.S0)

    def dry_call():
        # the flow cycle's call before its first Newton step: no element changes state on the
        # same initial state, so it is the device pass and the flags' download
        if wet:
            assert c.dry_rewet() == (0, 0)

    for w in range(a.warmup):
        reset()
        dry_call()
        st = c.newton_step(**opts)
        log(f"warmup {w}: {st.solve.iters} it, residual {st.solve.true_resid:.2e}, "
            f"{st.t_prepare + st.t_assemble + st.t_factor + st.t_solve + st.t_update:.2f}s")
    times, stats, t_dry = [], [], []
    c.kernel_stats(on=True)                     # HIP events around the kernel classes
    for k in range(a.steps):
        reset()
        t0 = time.perf_counter()
        dry_call()
        t_dry.append(time.perf_counter() - t0)
        st = c.newton_step(**opts)
        times.append(time.perf_counter() - t0)
        stats.append(st)
        log(f"step {k}: {times[-1]:.2f}s (assemble {st.t_assemble:.3f}, factor {st.t_factor:.3f}, "
            f"solve {st.t_solve:.2f}: {st.solve.iters} it, {st.solve.sweeps} sweeps, residual "
            f"{st.solve.true_resid:.2e})")
    ks = c.kernel_stats(on=False)
    T = sum(times) / len(times)
    last = stats[-1]
    its = max(last.solve.iters, 1)
    n_aggregates = c.aggregates()[1] if a.coarse != 0 else 0
    t_solve = sum(s.t_solve for s in stats) / len(stats)

    # kernel table: per class, launches and time per step, share of the step, algorithmic
    # bytes per launch and the fraction of the HBM peak they reach
    table = {}
    for name, (sec, byt, cnt) in ks.items():
        if cnt == 0:
            continue
        per = sec / a.steps
        avg = sec / cnt
        table[name] = {"kernel": KERNEL_NAMES[name], "launches_per_step": cnt / a.steps,
                       "avg_launch_ms": avg * 1e3, "ms_per_step": per * 1e3,
                       "share_of_step": per / T, "gb_per_launch": byt / cnt / 1e9,
                       "achieved_gb_s": byt / sec / 1e9, "frac_hbm_peak": byt / sec / HBM_PEAK}
    rest = T - sum(v["ms_per_step"] for v in table.values()) / 1e3
    table["other"] = {"kernel": "other kernels, host work and synchronisation",
                      "ms_per_step": rest * 1e3, "share_of_step": rest / T}
    dom = max((k for k in table if k != "other"), key=lambda k: table[k]["ms_per_step"])
    D = table[dom]
    byt = D["gb_per_launch"] * 1e9
    dur = D["avg_launch_ms"] / 1e3
    # HBM bytes per launch of the dominant kernel from the committed counter summary of the
    # same workload (rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE, calibrated on a device copy of
    # known size), used when the system and the kernel's algorithmic bytes match
    traffic = None
    tf = os.path.join(HERE, "profiles", "meander2M_hbm_traffic.json")
    if os.path.exists(tf) and dom in TRAFFIC_KEYS:
        rec = json.load(open(tf))
        k = rec.get("kernels", {}).get(TRAFFIC_KEYS[dom])
        if k and rec.get("n") == n and rec.get("nnz") == c.nnz and abs(k.get("algorithmic_bytes") - byt) < 1:
            traffic = k["traffic_bytes"]
    for name, v in table.items():
        if "avg_launch_ms" in v:
            log(f"kernel {name}: {v['launches_per_step']:.0f} launches, {v['avg_launch_ms']:.3f} ms avg, "
                f"{v['ms_per_step']:.0f} ms/step ({100 * v['share_of_step']:.0f}%), "
                f"{v['achieved_gb_s']:.0f} GB/s ({v['frac_hbm_peak']:.3f} of peak)")
    log(f"other: {rest * 1e3:.0f} ms/step")

    # learned leg: the same Newton step with the network correcting the two-level
    # preconditioner (same Krylov method, restart and refinement), one untimed and one timed
    learned, learned_reason = None, None
    if os.path.exists(a.learned):
        theta = np.load(a.learned)
        c.mpnn_set_weights(theta)
        lopts = dict(opts, precond=R.PREC_MPNN)
        for k in range(2):
            reset()
            t0 = time.perf_counter()
            dry_call()
            st = c.newton_step(**lopts)
            tl = time.perf_counter() - t0
            log(f"learned {'warmup' if k == 0 else 'step'}: {tl:.2f}s ({st.solve.iters} it, "
                f"{st.solve.sweeps} sweeps, fallback {st.solve.fallback}, residual "
                f"{st.solve.true_resid:.2e})")
        learned = {"weights": os.path.relpath(a.learned, HERE), "s_per_newton_step": tl,
                   "converged": bool(st.solve.converged), "true_resid": st.solve.true_resid,
                   "krylov_iters": st.solve.iters, "refine_sweeps": st.solve.sweeps,
                   "fallback": st.solve.fallback, "t_solve_s": st.t_solve,
                   "vs_two_level_step": tl / T,
                   "krylov_iters_two_level": last.solve.iters}
        if a.mkyrl != 30:
            # both preconditioners inside FGMRES(30) as well (the first step allocates the
            # longer basis and is not timed)
            f30 = {}
            for name, pk, reps in (("two_level", opts["precond"], 2), ("learned", R.PREC_MPNN, 1)):
                for k in range(reps):
                    reset()
                    t0 = time.perf_counter()
                    dry_call()
                    st = c.newton_step(**dict(opts, precond=pk, mkyrl=30))
                    t30 = time.perf_counter() - t0
                f30[name] = {"s_per_newton_step": t30, "krylov_iters": st.solve.iters,
                             "converged": bool(st.solve.converged), "fallback": st.solve.fallback}
                log(f"FGMRES(30) {name}: {t30:.2f}s ({st.solve.iters} it, fallback "
                    f"{st.solve.fallback}, residual {st.solve.true_resid:.2e})")
            learned["fgmres30"] = f30
    else:
        learned_reason = f"no trained weights at {a.learned}"

    # plain FP64 path on the 2M system (state reset, friction and inlet recomputed):
    # reference-order ILU(0), BiCGStab, bounded
    c.state_upload(d.U0, d.V0, d.S0)
    dry_call()
    c.prepare()
    c.assemble(R.F64)
    c.scale_l2()
    t0 = time.perf_counter()
    c.ilu0_factor(R.F64)
    t_fac64 = time.perf_counter() - t0
    out = c.solve(R.BICGSTAB, R.F64, R.PREC_ILU0, max_iter=a.plain_iters, eps=1e-8)
    plain_it = out.seconds / max(out.iters, 1)
    plain_elapsed = t_fac64 + out.seconds
    log(f"plain FP64 (2M): factor {t_fac64:.2f}s, {out.iters} BiCGStab it in {out.seconds:.2f}s "
        f"({plain_it:.3f} s/it), residual {out.accuracy:.2e}")
    c.close()

    cmp = None
    if a.cmp_along > 0:
        cmp = comparison(R, a)
        if cpu:
            cpu["dof_iters_per_s"] = cmp["n_eq"] * cpu["iters"] / cpu["value"]
            cmp["reference_cpu"] = {"s_per_newton_step": cpu["value"], "cores": 1,
                                    "krylov_iters": cpu["iters"],
                                    "accuracy_reached": cpu.get("accuracy"),
                                    "dof_iters_per_s": cpu["dof_iters_per_s"]}

    line = {
        "metric": METRIC,
        "value": T,
        "unit": "s per Newton step",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": T * 1e3,
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32+f64",
        "data": "synthetic",
        "config": {"workload": f"meander channel {a.n_along}x{a.n_across} cells, "
                               f"{d.n_elems} Taylor-Hood triangles, {n} equations, {c.nnz} nnz; "
                               "Newton step 1 from the initial state" +
                               (f"; floodplains rising {a.plain_rise:g} m/m, "
                                f"{wet['dry_elements']} elements dry and "
                                f"{wet['marsh_elements']} marsh after drying and rewetting "
                                f"(method 2, {wet['equations_all_wet']} equations when all wet)"
                                if wet else ""),
                   "solver": f"FGMRES({a.mkyrl}), FP32 matrix, coarse correction "
                             f"({n_aggregates} U,V,H aggregates over the strips' coarse "
                             f"segments, block cyclic reduction on the device) + strip ILU(0) ({a.strips or '2 per CU'} "
                             f"strips x {a.segments or 'about 560-row'} segments, dataflow "
                             f"factorisation), FP64 "
                             f"iterative refinement to 1e-8 (inner tolerance {a.eps:g}; a "
                             f"sweep that stalls hands the remaining ones to BiCGStab)",
                   "parallelism": "1 GPU"},
        "converged": bool(last.solve.converged),
        "true_resid": last.solve.true_resid,
        "krylov_iters": last.solve.iters,
        "refine_sweeps": last.solve.sweeps,
        "fallback": last.solve.fallback,
        "t_factor_s": last.t_factor,
        "t_solve_s": last.t_solve,
        "newton_steps_per_s": 1.0 / T,
        "krylov_gdof_iters_per_s": n * its / t_solve / 1e9,
        "kernels": table,
        "roofline": {"kernel": D["kernel"], "bound": "hbm", "achieved": D["achieved_gb_s"],
                     "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": D["frac_hbm_peak"],
                     "traffic": traffic, "algorithmic_bytes": byt, "avg_launch_ms": dur * 1e3,
                     "share_of_step": D["share_of_step"]},
        "drying": wet and dict(wet, dry_call_s=sum(t_dry) / len(t_dry)),
        "comparison": cmp,
        "plain_fp64_2M": {"factor_s": t_fac64, "s_per_bicgstab_iter": plain_it,
                          "iters_run": out.iters, "residual_reached": out.accuracy,
                          "elapsed_s": plain_elapsed, "converged": bool(out.converged),
                          # not at 1e-8 when stopped: its time to 1e-8 exceeds elapsed_s
                          "speedup_lower_bound": (plain_elapsed / T) if (last.solve.converged and
                                                                          not out.converged) else None},
        # value is the two-level path's step; the learned leg is timed beside it
        "learned": learned,
        "learned_reason": learned_reason,
        "cpu_baseline": cpu and {k: cpu[k] for k in ("value", "unit", "cores", "kind", "sample",
                                                      "dof_iters_per_s") if k in cpu},
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
