"""Triangular sweeps on the GPU at the edges of their layouts, against the oracle's ILU(0)
factors and triangular solves.

The sweeps sum a row's products in another order than the oracle, in FP64: each sum of w
products is off by at most about w 1.1e-16 of its terms' magnitude, and the systems here are
diagonally dominant (or the channel's, whose sweeps the other tests hold to the same bound),
so results agree within 1e-12 of the largest.
"""
import numpy as np
import pytest

from helpers import golden_deck, load_golden
from oracle import pyoracle as po
from rismo2d_amd import rmx

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = rmx.Context(0)
    yield c
    c.close()


def _band_csr(n, offsets, seed):
    """n rows, row i coupled to i - o and i + o for every offset o (a symmetric pattern), in
    random order after the diagonal; diagonally dominant."""
    rng = np.random.default_rng(seed)
    rp, cols, vals = [0], [], []
    for i in range(n):
        js = np.asarray([j for o in offsets for j in (i - o, i + o) if 0 <= j < n], int)
        js = rng.permutation(js)
        v = rng.standard_normal(len(js))
        cols += [i] + js.tolist()
        vals += [np.abs(v).sum() + 1.0] + v.tolist()
        rp.append(len(cols))
    return np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals)


# one block: entries per row and triangle at the edges of a lane's group (4), of a slot (16)
# and of 2, 4 and 8 slots (32, 64, 127), chains and independent rows
@pytest.mark.parametrize("n,width,stride", [(1, 0, 1), (2, 1, 1), (3, 2, 1), (17, 4, 3), (64, 0, 1),
                                            (65, 5, 7), (200, 16, 2), (300, 17, 11), (513, 32, 3),
                                            (700, 33, 5), (900, 63, 1), (65, 64, 1), (128, 127, 1),
                                            (2047, 13, 31)])
def test_single_block_of_single_rows(ctx, n, width, stride):
    print(f"[gpu] one block, {n} rows, {width} entries a side", flush=True)
    rp, cols, vals = _band_csr(n, [1 + stride * k for k in range(width)], 11)
    b = np.random.default_rng(12).standard_normal(n)
    ctx.csr_upload(rp, cols, vals, b)
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.ilu0_factor(prec)
        L, r = po.ilu0_factor(rp, cols, vals.astype(dt))
        assert r == 0
        ref = po.ilu0_solve(rp, cols, L, b)
        ctx.kernel_stats(True)
        y = ctx.ilu0_apply(b, prec)
        assert ctx.kernel_stats(False)["sweeps_block"][2] == 1
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec


# 61 and 256 waves for 128 and 300 segments: one to three blocks of a strip share a wave
@pytest.mark.parametrize("strips,segments", [(17, 128), (4, 300)])
def test_blocks_that_share_a_wave(ctx, strips, segments):
    print(f"[gpu] {strips} strips x {segments} segments, blocks sharing waves", flush=True)
    g = load_golden("channel200x20")
    ctx.upload_mesh(golden_deck(g))
    ctx.prepare()
    ctx.set_strips(strips, segments)
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    rp, cols = ctx.pattern()
    A, B = ctx.matrix(rmx.F64)
    block = ctx.blocks()
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    keep = block[rows] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=len(rp) - 1))])
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        L, _ = po.ilu0_factor(rp, cols, A.astype(dt))
        ref = po.ilu0_solve(rp2.astype(np.int32), cols[keep], L[keep], B)
        y = ctx.silu0_apply(B, prec)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec
    ctx.set_strips(0, 0)


# systems past one block (2,047 rows): chains and wide levels, one to four waves, entries per
# row and triangle at the edges of a slot (16) and of 2 and 4 slots; rows in units of 3 (one
# set of columns) and alone; the last keeps 21,000 rows alive, more than LDS holds (the staged
# level sweeps)
@pytest.mark.parametrize("n,width,stride,run", [(2048, 1, 1, 1), (2050, 3, 700, 1), (2500, 16, 1, 1),
                                                (3001, 17, 37, 1), (2100, 33, 2, 1), (6000, 4, 500, 3),
                                                (2049, 0, 1, 1), (9000, 2, 2000, 3),
                                                (45000, 2, 21000, 1)])
def test_single_strip_node_sweeps(ctx, n, width, stride, run):
    print(f"[gpu] one strip, {n} rows in runs of {run}, {width} entries a side", flush=True)
    rp, cols, vals = _band_csr(n // run, [1 + stride * k for k in range(width)], 21)
    if run > 1:                              # every row and column `run` times
        m, rng = n // run, np.random.default_rng(22)
        rp0, c0, rp, cols, vals = rp, cols, [0], [], []
        for i in range(m):
            js = (run * c0[rp0[i]:rp0[i + 1], None] + np.arange(run)).ravel()
            for r in range(run * i, run * i + run):
                o = rng.permutation(js[js != r])
                v = rng.standard_normal(len(o))
                cols += [r] + o.tolist()
                vals += [np.abs(v).sum() + 1.0] + v.tolist()
                rp.append(len(cols))
        rp, cols, vals = np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals)
    n = len(rp) - 1
    b = np.random.default_rng(12).standard_normal(n)
    ctx.csr_upload(rp, cols, vals, b)
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.ilu0_factor(prec)
        L, r = po.ilu0_factor(rp, cols, vals.astype(dt))
        assert r == 0
        ref = po.ilu0_solve(rp, cols, L, b)
        ctx.kernel_stats(True)
        y = ctx.ilu0_apply(b, prec)
        ran = ctx.kernel_stats(False)
        assert ran["sweep_lower"][2] == 1 and ran["sweep_upper"][2] == 1
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec


def _two_level_reference(ctx, prec, dt, r):
    """z = z1 + M^-1 (r - A z1), z1 = P (R A P)^-1 R r, in numpy with the oracle's ILU(0)."""
    import scipy.sparse as sp
    n = ctx.n
    rp, cols = ctx.pattern()
    A, _ = ctx.matrix(rmx.F64)
    agg, nc = ctx.aggregates()
    block = ctx.blocks()
    P = sp.csr_matrix((np.ones(n), (np.arange(n), agg)), shape=(n, nc))
    Ap = A.astype(dt)
    M = sp.csr_matrix((Ap.astype(np.float64), cols, rp), shape=(n, n))
    z1 = P @ np.linalg.solve((P.T @ M @ P).toarray(), P.T @ r)
    rows = np.repeat(np.arange(n), np.diff(rp))
    keep = block[rows] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))])
    L, _ = po.ilu0_factor(rp, cols, Ap)
    return z1 + po.ilu0_solve(rp2.astype(np.int32), cols[keep], L[keep], r - M @ z1)


# strips of less than a column of cells (the coarse matrix couples strips two apart), with few
# and many coarse unknowns a strip; one strip; a number of blocks that is no power of two.
# The same 1e-9 as the two-level test on the channel.
@pytest.mark.parametrize("nx,ny,strips,cseg", [(14, 250, 0, 2), (14, 250, 0, 20), (6, 60, 0, 5),
                                               (14, 250, 3, 8), (30, 130, 0, 6)])
def test_two_level_on_thin_strips(ctx, nx, ny, strips, cseg):
    from rismo2d_amd import deck as dk
    d = dk.meander(nx, ny, reach=3.125 * nx)
    ctx.set_coarse(cseg)
    ctx.set_strips(strips, 0)
    ctx.upload_mesh(d)
    ctx.time_step(30.0, 0.7, first=True)
    n = ctx.prepare()
    print(f"[gpu] two-level apply on a {nx} x {ny} meander, {n} equations, "
          f"{ctx.aggregates()[1]} coarse unknowns", flush=True)
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    r = np.random.default_rng(3).standard_normal(n)
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        ctx.coarse_factor(prec)
        ref = _two_level_reference(ctx, prec, dt, r)
        for _ in range(3):                   # the second and third apply meet used words
            y = ctx.precond_apply(rmx.PREC_SILU0C, r, prec)
            assert np.abs(y - ref).max() <= 1e-9 * np.abs(ref).max(), prec
    ctx.set_coarse(-1)
    ctx.set_strips(0, 0)


# blocks of up to 32, 64 and more coarse unknowns in the product with the inverse; the largest
# system that takes it (3,060 of 3,072 rows) and the next one (3,264), which takes the chain
@pytest.mark.parametrize("ny,strips,cseg", [(130, 6, 6), (130, 5, 15), (130, 7, 30), (260, 0, 15),
                                            (260, 0, 16)])
def test_two_level_inverse_and_chain(ctx, ny, strips, cseg):
    test_two_level_on_thin_strips(ctx, 60, ny, strips, cseg)


# factorisation by units: runs of 2 and 3 rows with one set of columns, longer runs (units of 3
# and a rest), one dense block; 62 to 68 and 123 to 128 columns (one and two columns a lane);
# `zero`: rows inside and at the ends of units whose diagonal and lower entries are zero, so
# that their pivots are repaired.  As for the row-by-row kernel: FP32 factors the oracle's
# bits, FP64 ones to 1e-12.
@pytest.mark.parametrize("n,width,stride,run,zero", [
    (2, 0, 1, 2, ()), (3, 0, 1, 3, ()), (4, 0, 1, 4, ()), (64, 0, 1, 64, ()), (65, 0, 1, 65, ()),
    (128, 0, 1, 128, ()), (600, 15, 2, 2, ()), (600, 16, 3, 2, ()), (500, 31, 1, 2, ()),
    (900, 10, 2, 3, ()), (900, 20, 1, 3, ()), (800, 8, 3, 4, ()), (600, 15, 1, 4, ()),
    (3000, 4, 7, 3, ()), (900, 4, 2, 3, (6, 10, 14, 300, 301, 898)), (600, 16, 1, 2, (1, 100, 598))])
def test_factorisation_by_units(ctx, n, width, stride, run, zero):
    print(f"[gpu] factorisation of {n} rows in runs of {run}, {width} runs a side", flush=True)
    rp0, c0, _ = _band_csr(n // run, [1 + stride * k for k in range(width)], 31)
    rng = np.random.default_rng(32)
    rp, cols, vals = [0], [], []
    for i in range(n // run):
        js = (run * c0[rp0[i]:rp0[i + 1], None] + np.arange(run)).ravel()
        for r in range(run * i, run * i + run):
            o = rng.permutation(js[js != r])
            v = rng.standard_normal(len(o))
            d = np.abs(v).sum() + 1.0
            if r in zero:
                d, v = 0.0, np.where(o < r, 0.0, v)
            cols += [r] + o.tolist()
            vals += [d] + v.tolist()
            rp.append(len(cols))
    rp, cols, vals = np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals)
    ctx.csr_upload(rp, cols, vals, np.ones(len(rp) - 1))
    L64, rep = po.ilu0_factor(rp, cols, vals)
    L32, _ = po.ilu0_factor(rp, cols, vals.astype(np.float32))
    assert (rep > 0) == (len(zero) > 0)
    ctx.ilu0_factor(rmx.F64)
    np.testing.assert_allclose(ctx.factors(rmx.F64), L64, rtol=1e-12, atol=1e-14)
    ctx.convert(rmx.F32)
    for _ in range(2):                       # the second pass meets flags of the first
        ctx.ilu0_factor(rmx.F32)
        np.testing.assert_array_equal(ctx.factors(rmx.F32), L32)


# the Gram-Schmidt kernels: sizes around a quad of entries and a workgroup's 1,024, one and two
# rounds of 512 workgroups, up to 8, 16 and 30 vectors.  A's diagonal exceeds its row's sum by 1,
# so |A^-1| <= 1 and the error is at most the residual, eps |b|; twice that for rounding.
@pytest.mark.parametrize("n,mkyrl", [(1, 3), (2, 5), (3, 7), (4, 7), (5, 15), (1023, 15), (1024, 30),
                                     (1025, 30), (2050, 15), (4099, 30), (60001, 15), (524287, 15),
                                     (524289, 30)])
def test_fgmres_on_ragged_sizes(ctx, n, mkyrl):
    import scipy.sparse as sp
    from scipy.sparse.linalg import splu
    print(f"[gpu] FGMRES({mkyrl}), {n} equations", flush=True)
    rng = np.random.default_rng(41)
    offs = [o for o in (1, 4, 9) if o < n]
    diags = [rng.standard_normal(n - o) for o in offs] + [rng.standard_normal(n - o) for o in offs]
    M = sp.diags(diags, offs + [-o for o in offs], shape=(n, n), format="csr") if offs else \
        sp.csr_matrix((n, n))
    d = np.asarray(abs(M).sum(axis=1)).ravel() + 1.0
    rows, cols, vals = sp.find(M)
    rows, cols = np.concatenate([np.arange(n), rows]), np.concatenate([np.arange(n), cols])
    vals = np.concatenate([d, vals])
    o = np.lexsort((cols, cols != rows, rows))           # the diagonal first in its row
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]).astype(np.int32)
    cols, vals = cols[o].astype(np.int32), vals[o]
    b = rng.standard_normal(n)
    ctx.csr_upload(rp, cols, vals, b)
    for prec, dt, eps in ((rmx.F64, np.float64, 1e-10), (rmx.F32, np.float32, 1e-5)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        out = ctx.solve(rmx.FGMRES, prec, rmx.PREC_NONE, max_iter=400, mkyrl=mkyrl, eps=eps)
        assert out.converged
        A = sp.csr_matrix((vals.astype(dt).astype(np.float64), cols, rp), shape=(n, n))
        x = splu(A.tocsc()).solve(b)
        assert np.abs(ctx.solution() - x).max() <= 2 * eps * np.linalg.norm(b), prec


# strip sweeps by chunks of 16 rows: blocks of one row, around one, three and four chunks (the
# loads ahead) and of 2,047 rows; rows of no, few (two packets), many (up to eight rounds) and
# more earlier entries than are loaded ahead (blocks of several strips: the two-level tests).  A sum of at most
# 128 products of FP64 values and inverses of diagonally dominant triangles (entries at most 1):
# 1e-12 as for the other sweeps.
@pytest.mark.parametrize("n,width,stride,strips", [
    (1, 0, 1, 1), (15, 3, 1, 1), (16, 3, 2, 1), (17, 3, 5, 1), (47, 2, 9, 1), (48, 5, 1, 1),
    (49, 0, 1, 1), (64, 8, 7, 1), (65, 20, 3, 1), (700, 10, 20, 1), (1024, 30, 17, 1),
    (1025, 50, 19, 1), (2047, 63, 17, 1), (2047, 4, 300, 1)])
def test_strip_sweeps_by_chunks(ctx, n, width, stride, strips):
    print(f"[gpu] {strips} strips, {n} rows, {width} entries a side", flush=True)
    rp, cols, vals = _band_csr(n, [1 + stride * k for k in range(width)], 51)
    b = np.random.default_rng(52).standard_normal(n)
    ctx.set_strips(strips, 0)
    ctx.csr_upload(rp, cols, vals, b)
    block = ctx.blocks()
    rows = np.repeat(np.arange(n), np.diff(rp))
    keep = block[rows] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        L, r = po.ilu0_factor(rp, cols, vals.astype(dt))
        assert r == 0
        ref = po.ilu0_solve(rp2, cols[keep], L[keep], b)
        y = ctx.precond_apply(rmx.PREC_SILU0, b, prec)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec
    ctx.set_strips(0, 0)


# the same strips cut into blocks of some ten rows: 3,400 (by chunks) and 3,740 (level by level);
# 1e-12 as for the other sweeps
@pytest.mark.parametrize("segments", [200, 220])
def test_strip_sweeps_of_many_blocks(ctx, segments):
    from rismo2d_amd import deck as dk
    d = dk.meander(30, 130, reach=93.75)
    ctx.set_strips(17, segments)
    ctx.upload_mesh(d)
    ctx.time_step(30.0, 0.7, first=True)
    n = ctx.prepare()
    block = ctx.blocks()
    print(f"[gpu] strip sweeps, {n} equations in {len(np.unique(block))} blocks", flush=True)
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    rp, cols = ctx.pattern()
    A, _ = ctx.matrix(rmx.F64)
    b = np.random.default_rng(61).standard_normal(n)
    rows = np.repeat(np.arange(n), np.diff(rp))
    keep = block[rows] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        L, _ = po.ilu0_factor(rp, cols, A.astype(dt))
        ref = po.ilu0_solve(rp2, cols[keep], L[keep], b)
        y = ctx.precond_apply(rmx.PREC_SILU0, b, prec)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec
    ctx.set_strips(0, 0)


# blocks whose neighbours have more chunks (the automatic cut of this mesh: 33 blocks, some of
# 703 rows before one of 705), after an apply of a vector of NaN to some 700 blocks that leaves
# them in the LDS of every compute unit; 1e-12 as for the other sweeps
def test_chunk_sweeps_after_nan_in_lds(ctx):
    from rismo2d_amd import deck as dk
    other = rmx.Context(0)
    systems = []
    for c, d in ((other, dk.meander(160, 320, reach=500.0)), (ctx, dk.meander(40, 64, reach=125.0))):
        c.upload_mesh(d)
        c.time_step(30.0, 0.7, first=True)
        n = c.prepare()
        c.assemble(rmx.F64)
        c.scale_l2()
        c.convert(rmx.F32)
        c.silu0_factor(rmx.F32)
        systems.append(n)
    rp, cols = ctx.pattern()
    A, _ = ctx.matrix(rmx.F64)
    block = ctx.blocks()
    rows, reach = rmx.chunk_reach(rp, cols, block)
    chunks = (rows + 15) // 16
    assert (reach <= 16 * chunks).all() and (chunks[1:] > chunks[:-1]).any()
    print(f"[gpu] strip sweeps, {systems[1]} equations in {len(rows)} blocks, after NaN in LDS", flush=True)
    L, _ = po.ilu0_factor(rp, cols, A.astype(np.float32))
    of = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    keep = block[of] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(of[keep], minlength=len(rp) - 1))]).astype(np.int32)
    b = np.random.default_rng(71).standard_normal(systems[1])
    ref = po.ilu0_solve(rp2, cols[keep], L[keep], b)
    for _ in range(3):
        y = other.precond_apply(rmx.PREC_SILU0, np.full(systems[0], np.nan), rmx.F32)
        assert np.isnan(y).all()
        y = ctx.precond_apply(rmx.PREC_SILU0, b, rmx.F32)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
    other.close()


# the sweeps that run where several could: blocks of the strip ILU(0) by chunks, by levels of
# nodes (RMX_SWEEP=2, or caps of their passes) or in stages (1); more rows a block than 2,047
@pytest.mark.parametrize("strips,segments,env,kind", [
    (17, 4, {}, "chunks"), (17, 4, {"RMX_SWEEP": "2"}, "blocks"), (17, 4, {"RMX_SWEEP": "1"}, "levels"),
    (17, 4, {"RMX_BLOCK_LEVEL_ROWS": "3"}, "blocks"), (17, 4, {"RMX_BLOCK_LEVEL_PAIRS": "5"}, "blocks"),
    (17, 220, {}, "blocks"), (1, 1, {}, "nodes"), (1, 1, {"RMX_SWEEP": "2"}, "nodes")])
def test_sweeps_that_run(ctx, strips, segments, env, kind, monkeypatch):
    for k in ("RMX_SWEEP", "RMX_BLOCK_LEVEL_ROWS", "RMX_BLOCK_LEVEL_PAIRS"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    ctx.upload_mesh(golden_deck(load_golden("channel200x20")))
    ctx.prepare()
    ctx.set_strips(strips, segments)
    assert ctx.sweeps() == kind
    ctx.set_strips(0, 0)


def _check_block_sweeps(ctx, strips, segments):
    """FP64 and FP32 applies of a channel's strip ILU(0) by block sweeps against the oracle's
    triangular solves of the block-restricted factors, 1e-12 as for the other sweeps."""
    ctx.upload_mesh(golden_deck(load_golden("channel200x20")))
    ctx.prepare()
    ctx.set_strips(strips, segments)
    assert ctx.sweeps() == "blocks"
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    rp, cols = ctx.pattern()
    A, B = ctx.matrix(rmx.F64)
    block = ctx.blocks()
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    keep = block[rows] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=len(rp) - 1))])
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        L, _ = po.ilu0_factor(rp, cols, A.astype(dt))
        ref = po.ilu0_solve(rp2.astype(np.int32), cols[keep], L[keep], B)
        y = ctx.silu0_apply(B, prec)
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max(), prec
    ctx.set_strips(0, 0)
    return block


# block sweeps of strips that the chunk sweeps take by default: a block a wave, and 61 and 256
# waves for 128 and 300 segments, two or more blocks of a strip sharing a wave
@pytest.mark.parametrize("strips,segments", [(17, 2), (17, 4), (4, 8), (4, 32), (17, 128), (4, 300)])
def test_block_sweeps_on_strips(ctx, strips, segments, monkeypatch):
    print(f"[gpu] block sweeps, {strips} strips x {segments} segments", flush=True)
    monkeypatch.setenv("RMX_SWEEP", "2")
    _check_block_sweeps(ctx, strips, segments)


# blocks that share waves of more than 2,047 rows, up to the most that the rule gives a wave (9/10
# of 4,093 rows on average): a strip's `segments` blocks cut into `groups` waves of neighbouring ones
@pytest.mark.parametrize("strips,segments,groups", [(2, 64, 5), (5, 4, 2), (5, 32, 2), (10, 16, 1),
                                                    (16, 128, 1)])
def test_block_sweeps_of_long_waves(ctx, strips, segments, groups, monkeypatch):
    print(f"[gpu] block sweeps, {strips} strips x {segments} segments in {groups} waves", flush=True)
    monkeypatch.setenv("RMX_SWEEP", "2")
    monkeypatch.setenv("RMX_BLOCK_WAVES", "1")
    block = _check_block_sweeps(ctx, strips, segments)
    rows = np.bincount(block // segments * groups + block % segments * groups // segments)
    assert len(rows) == strips * groups and 2047 < rows.max() <= 4093
    assert rows.mean() <= 0.9 * 4093


# the bytes reported for a launch are those of its system, however many were set up before
def test_reported_bytes_of_a_sweep(ctx, monkeypatch):
    monkeypatch.delenv("RMX_SWEEP", raising=False)
    ctx.upload_mesh(golden_deck(load_golden("channel200x20")))
    ctx.prepare()
    seen = []
    for strips, segments, kind in ((17, 4, "chunks"), (17, 220, "blocks"), (17, 4, "chunks"), (17, 4, "chunks"),
                                   (17, 220, "blocks"), (1, 1, "nodes")):
        ctx.set_strips(strips, segments)
        assert ctx.sweeps() == kind
        ctx.assemble(rmx.F64)
        ctx.scale_l2()
        _, B = ctx.matrix(rmx.F64)
        ctx.silu0_factor(rmx.F64)
        ctx.kernel_stats(True)
        ctx.silu0_apply(B, rmx.F64)
        seen.append(ctx.kernel_stats(False)["sweeps_block"][1])
    assert seen[0] > 0 and seen[1] > 0
    assert seen[2] == seen[3] == seen[0] and seen[4] == seen[1] and seen[5] == 0
    ctx.set_strips(0, 0)


# A coarse solve's bounded wait (one poll): every workgroup gives up and ends, the call reports
# it, and factored anew the apply is right again.  `caught`: the wait is given up inside a solve
# that ends with another error before it is reported; the factors still serve the next apply.
# 1e-9 as for the other two-level tests.
@pytest.mark.parametrize("caught", [False, True])
def test_coarse_wait_given_up(ctx, caught, monkeypatch):
    from rismo2d_amd import deck as dk
    ctx.set_coarse(16)
    ctx.set_strips(0, 0)
    ctx.upload_mesh(dk.meander(60, 260, reach=187.5))
    ctx.time_step(30.0, 0.7, first=True)
    n = ctx.prepare()
    print(f"[gpu] coarse solve with a wait of one poll, {n} equations, caught {caught}", flush=True)
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    r = np.random.default_rng(3).standard_normal(n)
    ctx.silu0_factor(rmx.F64)
    ctx.coarse_factor(rmx.F64)
    ref = ctx.precond_apply(rmx.PREC_SILU0C, r, rmx.F64)
    two = _two_level_reference(ctx, rmx.F64, np.float64, r)
    assert np.abs(ref - two).max() <= 1e-9 * np.abs(two).max()
    monkeypatch.setenv("RMX_COARSE_SPIN", "1")
    if caught:
        with pytest.raises(rmx.RmxError, match="proceed > 0 without a next solver"):
            ctx.solve(rmx.FGMRES, rmx.F64, rmx.PREC_SILU0C, max_iter=2, mkyrl=2, eps=1e-30, proceed=1)
    else:
        with pytest.raises(rmx.RmxError, match="wait for its neighbours"):
            ctx.precond_apply(rmx.PREC_SILU0C, r, rmx.F64)
        with pytest.raises(rmx.RmxError, match="not factored"):
            ctx.precond_apply(rmx.PREC_SILU0C, r, rmx.F64)
        ctx.coarse_factor(rmx.F64)
    monkeypatch.delenv("RMX_COARSE_SPIN")
    for _ in range(3):
        np.testing.assert_array_equal(ctx.precond_apply(rmx.PREC_SILU0C, r, rmx.F64), ref)
    ctx.set_coarse(-1)


# the factorisation's bounded wait (64 polls, with far more rows taken than can be ready): every
# wave gives up and ends, the call reports it, and the next factorisation has the oracle's bits;
# by units of three rows, and row by row (128 rows that are all coupled but for pairs, so that each
# is a unit, of more pivots than a unit takes)
@pytest.mark.parametrize("kind", ["units", "rows"])
def test_factorisation_wait_given_up(ctx, kind, monkeypatch):
    rng = np.random.default_rng(81)
    rp, cols, vals = [0], [], []
    n = 9000 if kind == "units" else 128
    for i in range(n):
        if kind == "units":
            js = np.arange(max(0, i // 3 - 4) * 3, min(n, (i // 3 + 5) * 3))
            js = js[js != i]
        else:
            js = np.arange(n)
            js = js[js % 64 != i % 64]
        v = rng.standard_normal(len(js))
        cols += [i] + js.tolist()
        vals += [np.abs(v).sum() + 1.0] + v.tolist()
        rp.append(len(cols))
    rp, cols, vals = np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals)
    print(f"[gpu] factorisation by {kind} with a wait of 64 polls, {n} rows", flush=True)
    ctx.csr_upload(rp, cols, vals, np.ones(n))
    ctx.convert(rmx.F32)
    monkeypatch.setenv("RMX_ILU_SPIN", "32")
    monkeypatch.setenv("RMX_ILU_WAVES", "4096")
    with pytest.raises(rmx.RmxError, match="wait for its pivot rows"):
        ctx.ilu0_factor(rmx.F32)
    monkeypatch.delenv("RMX_ILU_SPIN")
    monkeypatch.delenv("RMX_ILU_WAVES")
    L, _ = po.ilu0_factor(rp, cols, vals.astype(np.float32))
    for _ in range(2):
        ctx.ilu0_factor(rmx.F32)
        np.testing.assert_array_equal(ctx.factors(rmx.F32), L)


def _ilu0(n, rows):
    """ILU(0) of rows {column: value}, row by row; (lower multipliers, upper rows)."""
    low, up = [], []
    for i in range(n):
        a = dict(rows[i])
        for k in sorted(c for c in a if c < i):
            a[k] /= up[k][k]
            for c, u in up[k].items():
                if c > k and c in a:
                    a[c] -= a[k] * u
        low.append({c: v for c, v in a.items() if c < i})
        up.append({c: v for c, v in a.items() if c >= i})
    return low, up


def _ilu0_solve(low, up, b):
    x = np.array(b, float)
    for i in range(len(x)):
        x[i] -= sum(v * x[c] for c, v in low[i].items())
    for i in range(len(x) - 1, -1, -1):
        x[i] = (x[i] - sum(v * x[c] for c, v in up[i].items() if c > i)) / up[i][i]
    return x


# a caller's CSR rows as they may come: columns in any order, a pattern that is not symmetric,
# entries of value zero, a lower column twice in a row (its values add up, as in a product);
# one block (block and chunk sweeps) and more rows than a block takes (node sweeps).  Diagonally
# dominant; sums of some ten products and quotients in FP64: 1e-12 as for the other sweeps.
@pytest.mark.parametrize("form", ["asymmetric", "zeros", "repeated", "repeated runs"])
@pytest.mark.parametrize("n", [12, 300, 3000])
def test_csr_row_forms(ctx, n, form):
    print(f"[gpu] {n} CSR rows, {form}", flush=True)
    rng = np.random.default_rng(91)
    run = 3 if form == "repeated runs" else 1
    near = [np.unique(np.clip(i // run + rng.integers(-9, 10, 5), 0, n // run - 1)) for i in range(0, n, run)]
    if form != "asymmetric":
        near = [np.unique(np.concatenate([near[i], [j for j in range(len(near)) if abs(i - j) < 10 and i in near[j]],
                                          [i]])).astype(int) for i in range(len(near))]
    rows, rp, cols, vals = [], [0], [], []
    for i in range(n):
        js = [run * int(j) + q for j in near[i // run] for q in range(run) if run * j + q != i]
        v = rng.standard_normal(len(js))
        if form == "zeros":
            v *= rng.random(len(js)) < 0.6
        rows.append({i: float(np.abs(v).sum() + 1.0), **{j: float(x) for j, x in zip(js, v)}})
        ent = list(zip(js, v))
        if form.startswith("repeated"):
            part = rng.random(len(js))
            ent = [(j, x * p if j < i else x) for (j, x), p in zip(ent, part)] + \
                [(j, x - x * p) for (j, x), p in zip(ent, part) if j < i]
        o = rng.permutation(len(ent))
        cols += [i] + [ent[k][0] for k in o]
        vals += [rows[i][i]] + [ent[k][1] for k in o]
        rp.append(len(cols))
    rp, cols, vals = np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals, float)
    b = rng.standard_normal(n)
    ref = _ilu0_solve(*_ilu0(n, rows), b)
    ctx.set_strips(1, 0)
    ctx.csr_upload(rp, cols, vals, b)
    ctx.ilu0_factor(rmx.F64)
    ctx.silu0_factor(rmx.F64)
    for y in (ctx.ilu0_apply(b, rmx.F64), ctx.precond_apply(rmx.PREC_SILU0, b, rmx.F64)):
        assert np.abs(y - ref).max() <= 1e-12 * np.abs(ref).max()
    ctx.set_strips(0, 0)


# BiCGStab where the preconditioner solves the system exactly: a diagonal and small dense systems
# whose factors' solve leaves s = 0 to the last bit.  Diagonally dominant: |A^-1| <= 1, and x is off
# by at most some ten roundings of its terms.
@pytest.mark.parametrize("n,dense", [(1, False), (2, True), (3, True), (5, False), (12, True), (300, False),
                                     (5000, False)])
@pytest.mark.parametrize("seed", [0, 1, 2, 3])
def test_bicgstab_with_an_exact_preconditioner(ctx, n, dense, seed):
    print(f"[gpu] BiCGStab, {n} rows, exact preconditioner", flush=True)
    rng = np.random.default_rng(seed)
    A = np.zeros((n, n)) if dense else None
    rp, cols, vals = [0], [], []
    for i in range(n):
        js = rng.permutation([j for j in range(n) if j != i]) if dense else np.zeros(0, int)
        v = rng.standard_normal(len(js))
        cols += [i] + [int(j) for j in js]
        vals += [float(np.abs(v).sum() + 1.0 + rng.random())] + v.tolist()
        rp.append(len(cols))
    rp, cols, vals = np.asarray(rp, np.int32), np.asarray(cols, np.int32), np.asarray(vals, float)
    b = rng.standard_normal(n)
    ctx.csr_upload(rp, cols, vals, b)
    ctx.ilu0_factor(rmx.F64)
    out = ctx.solve(rmx.BICGSTAB, rmx.F64, rmx.PREC_ILU0, max_iter=20, eps=1e-12)
    if dense:
        A[np.repeat(np.arange(n), np.diff(rp)), cols] = vals
        x = np.linalg.solve(A, b)
    else:
        x = b / vals
    assert out.converged
    assert np.abs(ctx.solution() - x).max() <= 1e-12 * np.abs(b).max()


# what is told of a system's sweeps is the same whichever run: entries and levels of the packed level
# sweeps (RMX_SWEEP=1) and of the others, whose set-up has no use for levels
@pytest.mark.parametrize("strips,segments", [(0, 0), (1, 1), (5, 3), (17, 220)])
def test_sweep_info_of_every_kind(ctx, strips, segments, monkeypatch):
    ctx.upload_mesh(golden_deck(load_golden("channel200x20")))
    ctx.prepare()
    seen = {}
    for sweep in ("1", None):
        monkeypatch.setenv("RMX_SWEEP", sweep) if sweep else monkeypatch.delenv("RMX_SWEEP", raising=False)
        ctx.set_strips(strips, segments)
        assert (ctx.sweeps() == "levels") == (sweep == "1")
        for kind in (rmx.PREC_ILU0, rmx.PREC_SILU0):
            i = ctx.sweep_info(kind)
            seen[sweep, kind] = (i.lower_entries, i.upper_entries, i.lower_levels, i.upper_levels, i.strips,
                                 i.segments)
            assert min(seen[sweep, kind]) > 0
            assert ctx.sweep_info(kind).upper_levels == i.upper_levels
    for kind in (rmx.PREC_ILU0, rmx.PREC_SILU0):
        assert seen["1", kind] == seen[None, kind]
    ctx.set_strips(0, 0)


# a right-hand side with an infinity or a NaN: it reaches the rows that depend on it, as in the
# oracle's triangular solves, and the others keep their values (1e-12 as for the other sweeps):
# groups of rows coupled among themselves (5 within a chunk, 40 over several), and a channel
@pytest.mark.parametrize("group,width", [(1, 0), (5, 2), (40, 6), (23, 9)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_chunk_sweeps_of_non_finite_vectors(ctx, group, width, bad):
    print(f"[gpu] strip sweeps, groups of {group} rows, {bad} in the right-hand side", flush=True)
    n = 700
    rp0, c0, v0 = _band_csr(n, [1 + k for k in range(width)], 95)
    rows = np.repeat(np.arange(n), np.diff(rp0))
    keep = rows // group == c0 // group
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    cols, vals = c0[keep], v0[keep]
    b = np.random.default_rng(96).standard_normal(n)
    b[[0, 17, 350, 359, 698]] = bad
    ctx.set_strips(1, 0)
    ctx.csr_upload(rp, cols, vals, np.ones(n))
    assert ctx.sweeps() == "chunks"
    for prec, dt in ((rmx.F64, np.float64), (rmx.F32, np.float32)):
        if prec == rmx.F32:
            ctx.convert(rmx.F32)
        ctx.silu0_factor(prec)
        L, _ = po.ilu0_factor(rp, cols, vals.astype(dt))
        ref = po.ilu0_solve(rp, cols, L, b)
        y = ctx.precond_apply(rmx.PREC_SILU0, b, prec)
        ok = np.isfinite(ref)
        assert ok.any() and not ok.all()
        np.testing.assert_array_equal(np.isfinite(y), ok)
        assert np.abs(y[ok] - ref[ok]).max() <= 1e-12 * np.abs(ref[ok]).max(), prec
    ctx.set_strips(0, 0)


def test_chunk_sweeps_of_non_finite_vectors_on_a_mesh(ctx):
    from rismo2d_amd import deck as dk
    ctx.upload_mesh(dk.channel(60, 13, length=300.0, width=65.0))
    ctx.time_step(30.0, 0.7, first=True)
    n = ctx.prepare()
    ctx.assemble(rmx.F64)
    ctx.scale_l2()
    ctx.silu0_factor(rmx.F64)
    assert ctx.sweeps() == "chunks"
    rp, cols = ctx.pattern()
    A, _ = ctx.matrix(rmx.F64)
    block = ctx.blocks()
    of = np.repeat(np.arange(n), np.diff(rp))
    keep = block[of] == block[cols]
    rp2 = np.concatenate([[0], np.cumsum(np.bincount(of[keep], minlength=n))]).astype(np.int32)
    L, _ = po.ilu0_factor(rp, cols, A)
    for row in (0, n // 3, n // 2 + 5, n - 1):
        b = np.random.default_rng(97).standard_normal(n)
        b[row] = np.nan
        ref = po.ilu0_solve(rp2, cols[keep], L[keep], b)
        y = ctx.precond_apply(rmx.PREC_SILU0, b, rmx.F64)
        ok = np.isfinite(ref)
        assert np.isfinite(y[ok]).all()
        assert np.abs(y[ok] - ref[ok]).max() <= 1e-12 * np.abs(ref[ok]).max()
