"""Layout of the strip sweeps by chunks of 16 rows (host code): what a block's loads name in LDS
lies among the block's own rows, also where they run ahead of its last chunk.  LDS past a
block's rows holds whatever ran before, and zero times a NaN is a NaN."""
import numpy as np
import pytest

from rismo2d_amd import deck as dk
from rismo2d_amd import rmx
from test_gpu_sweeps import _band_csr


def _inside(rp, cols, block):
    rows, reach = rmx.chunk_reach(rp, cols, block)
    assert rows.tolist() == np.bincount(block)[np.bincount(block) > 0].tolist()
    assert (reach <= (rows + 15) // 16 * 16).all(), (rows, reach)


# entries a side from none to 24 and strides within and past a chunk: chunks of one to six
# packets, two and four of them loaded ahead; blocks of one row, of a few chunks and of 2,047
# rows, before and after larger and smaller ones
@pytest.mark.parametrize("width,stride", [(0, 1), (2, 1), (3, 17), (8, 17), (9, 16), (10, 5), (12, 3),
                                          (20, 17), (24, 2)])
@pytest.mark.parametrize("sizes", [(1, 200), (16, 17, 700, 1), (560, 640), (703, 705), (40, 2047, 30, 900),
                                   (300, 364, 428, 492, 16, 1000)])
def test_loads_stay_inside_their_block(width, stride, sizes):
    rp, cols, _ = _band_csr(sum(sizes), [1 + stride * k for k in range(width)], 3)
    _inside(rp, cols, np.repeat(np.arange(len(sizes)), sizes))


def _mesh_pattern(d):
    """Pattern of a mesh's system and the node of every equation, from the oracle's numbering."""
    from oracle import pyoracle as po
    m = po.OracleModel(d)
    m.prepare()
    rp, cols = m.pattern()
    eq = m.numbering().reshape(-1)
    group = np.zeros(len(rp) - 1, np.int64)
    group[eq[eq >= 0]] = np.nonzero(eq >= 0)[0] // 3
    return rp, cols, group


# a channel of triangles, one of eight-node quadrilaterals and a meander, cut into ranges of rows
# that start with a node, of 300 to 900 rows
@pytest.mark.parametrize("kind", ["triangles", "quads", "meander"])
def test_loads_stay_inside_their_block_on_meshes(kind):
    d = dk.meander(50, 40, reach=156.25) if kind == "meander" else \
        dk.channel(60, 13, length=300.0, width=65.0, quads=kind == "quads")
    rp, cols, group = _mesh_pattern(d)
    n = len(rp) - 1
    first = np.nonzero(np.concatenate([[True], group[1:] != group[:-1]]))[0]
    rng = np.random.default_rng(5)
    cuts = np.cumsum(rng.integers(300, 900, 1 + n // 300))
    cuts = np.unique(first[np.searchsorted(first, cuts[cuts < n - 3])])
    _inside(rp, cols, np.searchsorted(cuts, np.arange(n), side="right"))
