"""Hermite data of edges that brushes touch, against the oracle bit for bit: op counts
around the wave's size, brushes that tie with each other, nearly flat, huge, inside out
and rotated ones, at chunks of few and of many edges, alone and in a batch (needs a GPU)."""
import numpy as np
import pytest

from leven_amd import mesher, workloads
from oracle import py_oracle

pytestmark = pytest.mark.gpu


def _ops(n, seed, voxels, scale):
    rng = np.random.default_rng(seed)
    ops, _ = workloads.make_ops(n, seed=seed, rotated=True, extent=voxels * scale,
                                y_range=(-0.4 * voxels * scale, 0.4 * voxels * scale),
                                size_range=(0.5 * scale, 0.2 * voxels * scale))
    for k in range(0, n, 5):
        ops[k] = ops[rng.integers(0, n)]  # the same brush again: every sample ties
    for k in range(1, n, 7):
        ops[k]["dims"][rng.integers(0, 3)] = 0.01  # nearly flat, or a sphere of no size
    if n > 2:
        ops[2]["dims"][:3] = 3.0 * voxels * scale  # holds the whole chunk
    if n > 3:
        ops[3]["dims"][:3] = -1.0  # inside out: holds nothing
    return ops


@pytest.mark.parametrize("voxels,lod,n", [(4, 0, 1), (16, 0, 2), (16, 3, 40), (64, 0, 63), (64, 1, 65), (64, 0, 300)])
def test_brush_edges_match_oracle(voxels, lod, n):
    desc = workloads.terrain_desc()
    mesher.init(desc, 2, 0)
    mesher.clear_csg_ops()
    scale = 1 << lod
    size = 4 * voxels * scale
    mn = (0, -size // 2 // 4 * 4, 0)
    ops = _ops(n, 100 + n, voxels, scale)
    print(f"brush edges: N={voxels} lod={lod} ops={n}", flush=True)
    c = py_oracle.Chunk(voxels).generate(desc, py_oracle.perm_table(2), mn, size, ops=ops).build()
    ctx = mesher.Context(voxels)
    g = ctx.debug_stages(mn, size, ops)
    ids, data = c.edges()
    assert (g["edge_ids"] == ids).all()
    assert (g["edge_data"].view(np.uint32) == data.view(np.uint32)).all()
    # in a batch, between chunks without brushes
    for op in ops:
        mesher.store_csg_op(op, [mn[0], mn[1], mn[2]], [mn[0] + size, mn[1] + size, mn[2] + size])
    far = [(mn[0] + 40 * size, mn[1], mn[2]), mn, (mn[0] - 40 * size, mn[1], mn[2])]
    b = mesher.Batch(voxels, 3)
    b.set_chunks(far, [size] * 3)
    b.run()
    v, t, _ = b.get_mesh(1)
    mesher.clear_csg_ops()
    pos, nrm = c.positions()
    if len(t):
        assert (v["pos"].view(np.uint32) == pos.view(np.uint32)).all()
        assert (v["normal"].view(np.uint32) == nrm.view(np.uint32)).all()
    b.close()
    ctx.close()
