"""Performance cases: the work that programs on this library have it do, through
``rismo2d_amd.rmx.Context`` and ``rismo2d_amd.run``.

* ``newton``: a state goes in, one Newton step runs (friction and inlet set-up, assembly,
  scaling, factorisation, Krylov solve, update), the new state comes out.  The two solver
  paths of ``rismo2d_amd.run``: ``plain`` (FP64 BiCGStab with the reference-order ILU(0), the
  default of ``newton_step``) and ``fast`` (FGMRES(15) on the FP32 matrix with the two-level
  preconditioner inside FP64 refinement).  ``dt`` > 0 is a step of the theta scheme, 0
  stationary flow; ``rise`` > 0 a reach whose outer floodplains are dry, with the flow
  cycle's drying call before the step; ``fresh`` a mesh that the context has not seen, its
  set-up included.
* ``flow``: a time loop under an inlet hydrograph, each time step iterated to the
  reference's convergence test.
* ``linearise``: the Newton system of a state (assembly, scaling) and one product with it.
* ``factor``: the reference's preconditioner for a caller with a Krylov loop of its own,
  ILU(0) factorisation and one application; ``two_level`` the same with the strip ILU(0) and
  the coarse space in FP32.
* ``csr``: a linear system that the caller keeps in CSR, factored and solved.
* ``train``: loss, gradient and forward pass of the learned preconditioner on a sample.

The solves run to 1e-11 (plain 1e-12), as the repository's comparisons with the reference's
records do, so that the state is determined to well below the Newton iteration's tolerance.
"""
from __future__ import annotations

import numpy as np

from rismo2d_amd import deck as dk
from rismo2d_amd import mpnn
from rismo2d_amd import rmx
from rismo2d_amd import run as rr

PLAIN = dict(rr.PLAIN, max_iter=2000)
FAST = dict(rr.FAST, refine_tol=1e-11, refine_max=20)
THETA = 0.7


def listed():
    return [
        # the repository's smallest deck: a user's first run, launches and synchronisations
        dict(name="newton_plain_20x4", kind="newton", mesh="channel", nx=20, ny=4, quads=False,
             turb=1, path="plain", dt=0.0, rise=0.0, fresh=False),
        # the straight 200 x 20 channel under the default solver, a time step of a flood
        dict(name="newton_plain_200x20", kind="newton", mesh="channel", nx=200, ny=20,
             quads=False, turb=1, path="plain", dt=30.0, rise=0.0, fresh=False),
        # the same channel, stationary flow on the fast path
        dict(name="newton_fast_200x20", kind="newton", mesh="channel", nx=200, ny=20,
             quads=False, turb=1, path="fast", dt=0.0, rise=0.0, fresh=False),
        # eight-node quadrilaterals with the algebraic eddy viscosity: a hydrograph's first
        # time steps, each a few Newton steps
        dict(name="flow_fast_quads_60x13", kind="flow", mesh="channel", nx=60, ny=13, quads=True,
             turb=2, path="fast", dt=20.0, steps=2),
        # the benchmark's comparison reach with its floodplains dried, one Newton step
        dict(name="newton_fast_dried_80x320", kind="newton", mesh="meander", nx=80, ny=320,
             quads=False, turb=1, path="fast", dt=30.0, rise=0.012, fresh=False),
        # the 204,800-triangle reach the learned preconditioner is trained on, all wet
        dict(name="newton_fast_320x320", kind="newton", mesh="meander", nx=320, ny=320,
             quads=False, turb=1, path="fast", dt=30.0, rise=0.0, fresh=False),
        # the largest: 409,600 triangles, 1.8 million equations
        dict(name="newton_fast_640x320", kind="newton", mesh="meander", nx=640, ny=320,
             quads=False, turb=1, path="fast", dt=30.0, rise=0.0, fresh=False),
        # a deck read for the first time, dried, and stepped: mesh, numbering, patterns, plans
        dict(name="newton_fresh_dried_41x63", kind="newton", mesh="meander", nx=41, ny=63,
             quads=False, turb=1, path="fast", dt=30.0, rise=0.012, fresh=True),
        # a drop-in caller's preconditioner on the comparison reach, FP64, reference order
        dict(name="factor_ilu0_80x320", kind="factor", mesh="meander", nx=80, ny=320,
             two_level=False),
        # a drop-in caller's own system: 30 x 333 points with three unknowns each
        dict(name="csr_plain_333x30", kind="csr", nx=333, ny=30, path="plain"),
        # the learned preconditioner's training step on a reach
        dict(name="train_40x160", kind="train", mesh="meander", nx=40, ny=160),
        # the Newton matrix of a vegetated channel with Elder's viscosity
        dict(name="linearise_400x101", kind="linearise", mesh="channel", nx=400, ny=101,
             quads=False, turb=211),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    pick = rng.random()
    if pick < 0.2:                           # plain path: channels up to about 200 x 20 cells
        nx, ny = _log_int(rng, 10, 200), _log_int(rng, 3, 20)
        return dict(kind="newton", mesh="channel", nx=nx, ny=ny, quads=rng.random() < 0.3,
                    turb=rng.choice([1, 2]), path="plain", dt=rng.choice([10.0, 30.0]), rise=0.0,
                    fresh=False)
    if pick < 0.35:                          # fast path on channels
        nx, ny = _log_int(rng, 10, 400), _log_int(rng, 3, 40)
        quads = rng.random() < 0.3
        return dict(kind="newton", mesh="channel", nx=nx, ny=ny, quads=quads,
                    turb=rng.choice([1, 2]), path="fast",
                    dt=rng.choice([10.0, 30.0]) if quads else rng.choice([0.0, 30.0]), rise=0.0,
                    fresh=False)
    if pick < 0.6:                           # fast path on meandering reaches
        nx, ny = _log_int(rng, 30, 400), _log_int(rng, 48, 320)
        return dict(kind="newton", mesh="meander", nx=nx, ny=ny, quads=False, turb=1,
                    path="fast", dt=rng.choice([10.0, 30.0]), rise=rng.choice([0.0, 0.012]),
                    fresh=rng.random() < 0.2 and nx * ny < 8000)
    if pick < 0.7:
        return dict(kind="flow", mesh="channel", nx=_log_int(rng, 12, 120),
                    ny=_log_int(rng, 3, 16), quads=rng.random() < 0.5, turb=rng.choice([1, 2]),
                    path="fast", dt=rng.choice([10.0, 20.0]), steps=rng.choice([1, 2]))
    if pick < 0.8:
        return dict(kind="factor", mesh="meander", nx=_log_int(rng, 20, 160),
                    ny=_log_int(rng, 40, 320), two_level=rng.random() < 0.5)
    if pick < 0.9:
        return dict(kind="csr", nx=_log_int(rng, 20, 400), ny=_log_int(rng, 4, 40),
                    path=rng.choice(["plain", "mixed"]))
    if pick < 0.95:
        return dict(kind="train", mesh="meander", nx=_log_int(rng, 20, 80),
                    ny=_log_int(rng, 40, 160))
    return dict(kind="linearise", mesh="channel", nx=_log_int(rng, 40, 400),
                ny=_log_int(rng, 10, 101), quads=rng.random() < 0.5,
                turb=rng.choice([1, 2, 211]))


def _deck(case, seed):
    nx, ny = case["nx"], case["ny"]
    if case["mesh"] == "meander":
        # the benchmark's resolution along the reach, the full width across
        return dk.meander(n_along=nx, n_across=ny, reach=10000.0 * nx / 3200, seed=seed,
                          plain_rise=case.get("rise", 0.0))
    turb = case["turb"]
    kw = dict(turb=turb, turb_seed=seed)
    if turb % 10 == 2:
        kw.update(turb_st=(0.5, 1.5))
    if turb // 10 % 10 == 1:
        kw.update(turb_estx=(0.4, 1.2), turb_esty=(0.05, 0.3))
    if case["kind"] == "linearise":
        kw.update(veg_frac=0.3, veg_band=0.3, veg_seed=seed)
    return dk.channel(nx, ny, length=5.0 * nx, width=5.0 * ny, noise_corr=10.0, seed=seed,
                      Q=2.5 * ny, quads=case["quads"], **kw)


def _csr(nx, ny, rng):
    """Three coupled unknowns per point of an nx x ny lattice, every point coupled to its
    eight neighbours (numbered across the width first, as a channel's equations are):
    convection along x, diffusion, friction-like coupling of a point's unknowns."""
    i, j = (a.ravel() for a in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))
    p = i * ny + j
    rows, cols, vals = [], [], []
    for di in (-1, 0, 1):
        for dj in (-1, 0, 1):
            ok = (i + di >= 0) & (i + di < nx) & (j + dj >= 0) & (j + dj < ny)
            a, b = p[ok], p[ok] + di * ny + dj
            for u in range(3):
                for v in range(3):
                    m = len(a)
                    if di == 0 and dj == 0:
                        w = (11.5 if u == v else 0.6) + 0.2 * rng.standard_normal(m)
                    else:
                        w = (-1.0 - 0.5 * (di == -1) if u == v else 0.0)
                        w = w + 0.1 * rng.standard_normal(m)
                    rows.append(3 * a + u)
                    cols.append(3 * b + v)
                    vals.append(np.broadcast_to(w, (m,)))
    rows, cols, vals = (np.concatenate(t) for t in (rows, cols, vals))
    o = np.lexsort((cols, cols != rows, rows))       # the diagonal first in every row
    rows, cols, vals = rows[o], cols[o], vals[o]
    n = 3 * nx * ny
    rowptr = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rowptr[1:])
    x = rng.standard_normal(n)
    b = np.bincount(rows, weights=vals * x[cols], minlength=n)
    return rowptr.astype(np.int32), cols.astype(np.int32), vals, b, x


def prepare(case, seed):
    kind = case["kind"]
    ctx = rmx.Context(0)
    if kind == "csr":
        rowptr, cols, vals, b, _ = _csr(case["nx"], case["ny"], np.random.default_rng(seed))
        ctx.csr_upload(rowptr, cols, vals, b)
        if case["path"] == "mixed":
            ctx.convert(rmx.F32)
        return dict(case=case, ctx=ctx, b=b)
    d = _deck(case, seed)
    s = dict(case=case, ctx=ctx, deck=d)
    rng = np.random.default_rng(seed + 5)
    if kind in ("newton", "flow"):
        s["solve"] = PLAIN if case["path"] == "plain" else FAST
    if kind == "flow":
        s["hydrograph"] = [[0.0, d.Q_inlet, 2.1], [120.0, 1.5 * d.Q_inlet, 2.2]]
    if case.get("fresh"):
        return s
    ctx.upload_mesh(d)
    ctx.set_params()
    if kind in ("factor", "train"):
        ctx.time_step(30.0, THETA, first=True)
    ctx.prepare()
    if kind == "newton" and case["rise"] > 0.0:
        ctx.dry_rewet()
    if kind in ("factor", "train"):
        ctx.assemble(rmx.F64)
        ctx.scale_l2()
        s["b"] = rng.standard_normal(ctx.n)
    if kind == "factor" and case["two_level"]:
        ctx.convert(rmx.F32)
    if kind == "linearise":
        s["x"] = rng.standard_normal(ctx.n)
    if kind == "train":
        theta = mpnn.init_weights(seed % 1000)
        theta[-(mpnn.C + 1) * mpnn.O:] = 0.05 * rng.standard_normal((mpnn.C + 1) * mpnn.O)
        ctx.mpnn_set_weights(theta)
        ctx.mpnn_add_sample(s["b"], 1)
    return s


def run(s):
    case, c = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "newton":
        d = s["deck"]
        if case["fresh"]:
            c.upload_mesh(d)
            c.set_params()
        else:
            c.state_upload(d.U0, d.V0, d.S0)
        if case["dt"] > 0.0:
            c.time_step(case["dt"], THETA, first=True)
        if case["rise"] > 0.0:
            c.dry_rewet()
        c.newton_step(**s["solve"])
        return c.state()
    if kind == "flow":
        d = s["deck"]
        c.state_upload(d.U0, d.V0, d.S0)
        rr.time_loop(c, case["steps"], case["dt"], THETA, 8, lambda: c.newton_step(**s["solve"]),
                     hydrograph=s["hydrograph"])
        return c.state()
    if kind == "linearise":
        d = s["deck"]
        c.state_upload(d.U0, d.V0, d.S0)
        c.prepare()
        c.assemble(rmx.F64)
        return c.scale_l2(), c.spmv(s["x"], rmx.F64)
    if kind == "factor":
        if case["two_level"]:
            c.silu0_factor(rmx.F32)
            c.coarse_factor(rmx.F32)
            return c.precond_apply(rmx.PREC_SILU0C, s["b"], rmx.F32)
        c.ilu0_factor(rmx.F64)
        return c.ilu0_apply(s["b"], rmx.F64)
    if kind == "csr":
        c.set_rhs(s["b"])
        if case["path"] == "mixed":
            c.silu0_factor(rmx.F32)
            c.solve(**dict(FAST, precond=rmx.PREC_SILU0, refine_tol=1e-12))
        else:
            c.ilu0_factor(rmx.F64)
            c.solve(**PLAIN)
        return c.solution()
    loss, grad = c.mpnn_loss_grad(0)
    z, feat = c.mpnn_forward(s["b"])
    return loss, grad, z, feat


def exact(case, seed):
    """The solution of a caller's own system: its right-hand side is made from it."""
    if case["kind"] != "csr":
        return None
    return _csr(case["nx"], case["ny"], np.random.default_rng(seed))[4]


def work(case):
    """What one pass cannot do without: the state, mesh or vectors in and out, the system's
    values formed and used once, the element integrals."""
    cells = case["nx"] * case["ny"]
    if case["kind"] == "csr":
        nnz, n = 81.0 * cells, 3.0 * cells
        return {"bytes": 2 * 12 * nnz + 16 * n, "flops": 2 * nnz}
    quads = case.get("quads", False)
    elems = cells * (1 if quads else 2)
    nodes = cells * (3 if quads else 4)
    n = nodes * 2.25
    nnz = elems * (272.0 if quads else 133.0)
    element_flops = 40e3 if quads else 13.5e3
    mesh = elems * 32 + nodes * 24
    if case["kind"] == "factor":
        return {"bytes": 8 * nnz * 2 + 4 * nnz + 16 * n, "flops": 20 * nnz}
    if case["kind"] == "train":
        # six 128 x 64 layers per node, forward (twice: loss and forward pass), backward and
        # weight gradient; the activations written and read
        return {"bytes": 12 * nnz + nodes * 6 * 128 * 2 * 2, "flops": 4 * 2 * 128 * 64 * 6 * nodes}
    passes = 4 * case["steps"] if case["kind"] == "flow" else 1
    return {"bytes": passes * (mesh + 7 * 8 * nodes + 16 * nnz),
            "flops": passes * (element_flops * elems + 4 * nnz)}
