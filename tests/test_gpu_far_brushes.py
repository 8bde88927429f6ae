"""Brushes far from the origin, where FP32 cannot hold every voxel position: from 2^23 voxels
on the middle of an edge is rounded to one of its ends, and from 2^24 voxels on whole samples
are.  Materials, hermite data and meshes against the oracle bit for bit, in both forms of the
brush kernel (needs a GPU)."""
import numpy as np
import pytest

from leven_amd import mesher, workloads
from oracle import py_oracle

pytestmark = pytest.mark.gpu

N = 16


def _ops(n, x0, scale, seed):
    """Brushes over the chunk at x0, with centres on whole and half voxels where FP32 has them."""
    ops, _ = workloads.make_ops(n, seed=seed, rotated=True, extent=N * scale, y_range=(-6.0 * scale, 6.0 * scale),
                                size_range=(0.7 * scale, 5.0 * scale))
    for op in ops:
        op["origin"][0] = np.float32(x0) + np.float32(np.round(op["origin"][0]))
    return ops


@pytest.mark.parametrize("ops", [3, 40, 100])
@pytest.mark.parametrize("x0,lod", [((1 << 23) - 8, 0), (-(1 << 23) - 8, 0), ((1 << 23) + 1000, 0), ((1 << 23) - 16, 1),
                                    ((1 << 24) - 8, 0), ((1 << 24) + 1003, 0), (-(1 << 25) - 77, 0), ((1 << 26) + 5, 0),
                                    ((1 << 26) + 10, 1)])
def test_far_brushes_match_oracle(x0, lod, ops):
    desc = workloads.heightfield_desc()
    mesher.init(desc, 2, 0)
    mesher.clear_csg_ops()
    scale = 1 << lod
    size, mn = 4 * N * scale, (4 * x0, -2 * N * scale, 0)
    brushes = _ops(ops, x0, scale, 7 + ops)
    print(f"far brushes: x0={x0} lod={lod} ops={ops}", flush=True)
    c = py_oracle.Chunk(N).generate(desc, py_oracle.perm_table(2), mn, size, ops=brushes).build()
    ids, data = c.edges()
    assert len(ids) > 100
    ctx = mesher.Context(N)
    g = ctx.debug_stages(mn, size, brushes)
    assert (g["materials"] == c.materials()).all()
    assert len(g["edge_ids"]) == len(ids) and (g["edge_ids"] == ids).all()
    assert (g["edge_data"].view(np.uint32) == data.view(np.uint32)).all()
    ctx.close()
    # the scan of more than a few chunks: this one among eight without brushes
    for op in brushes:
        mesher.store_csg_op(op, mn, [v + size for v in mn])
    b = mesher.Batch(N, 9)
    b.set_chunks([(mn[0], mn[1] + 40 * size * k, mn[2]) for k in range(9)], [size] * 9)
    b.run()
    v, t, _ = b.get_mesh(0)
    b.close()
    mesher.clear_csg_ops()
    pos, nrm = c.positions()
    tri = c.triangles()
    assert len(t) == len(tri) > 0 and (t == tri).all()
    assert (v["pos"].view(np.uint32) == pos.view(np.uint32)).all()
    assert (v["normal"].view(np.uint32) == nrm.view(np.uint32)).all()


@pytest.mark.parametrize("axis,at", [(0, 28), (0, 27), (1, 25), (1, 26), (1, 27), (2, 26), (2, 27)])
def test_far_materials_match_oracle(axis, at):
    """Tiles of samples that round to few different positions, all air but for the brushes."""
    desc = workloads.heightfield_desc()
    mesher.init(desc, 2, 0)
    mesher.clear_csg_ops()
    ctx = mesher.Context(N)
    solid = 0
    for k in range(8):
        size, vox = 4 * N, [0, 64, 0]
        vox[axis] = (1 << at) + 16 * k + k
        brushes, _ = workloads.make_ops(30, seed=3 * at + k, extent=N, y_range=(0.0, 16.0), size_range=(0.5, 3.0))
        for op in brushes:
            op["type"], op["material"] = 0, 1
            for a in range(3):
                op["origin"][a] = np.float32(vox[a]) + np.float32(np.round(op["origin"][a]))
        mn = tuple(4 * v for v in vox)
        print(f"far materials: axis={axis} at=2^{at} {k}", flush=True)
        c = py_oracle.Chunk(N).generate(desc, py_oracle.perm_table(2), mn, size, ops=brushes)
        g = ctx.debug_stages(mn, size, brushes)
        assert (g["materials"] == c.materials()).all()
        solid += int((c.materials() == 1).sum())
    ctx.close()
    assert solid > 0


@pytest.mark.parametrize("axis,value", [(0, np.nan), (1, np.nan), (2, np.nan), (0, np.inf), (1, -np.inf), (2, 1e30)])
def test_brushes_without_a_place(axis, value):
    """A brush's distance ignores the axes along which its centre is no number."""
    desc = workloads.heightfield_desc()
    mesher.init(desc, 2, 0)
    mesher.clear_csg_ops()
    mn, size = (0, -2 * N, 0), 4 * N
    ops = _ops(40, 0, 1, 21)
    for k in (5, 17, 18, 33):
        ops[k]["origin"][axis] = value
        ops[k]["type"], ops[k]["material"] = k & 1, 2
        ops[k]["brush"], ops[k]["rotate_y"], ops[k]["dims"][:3] = 0, 0.7 * (k & 1), 1.5
    print(f"brushes without a place: axis={axis} {value}", flush=True)
    c = py_oracle.Chunk(N).generate(desc, py_oracle.perm_table(2), mn, size, ops=ops).build()
    ctx = mesher.Context(N)
    g = ctx.debug_stages(mn, size, ops)
    ctx.close()
    ids, data = c.edges()
    assert (g["materials"] == c.materials()).all()
    assert len(ids) == len(g["edge_ids"]) and (g["edge_ids"] == ids).all()
    same = (g["edge_data"].view(np.uint32) == data.view(np.uint32)) | (np.isnan(g["edge_data"]) & np.isnan(data))
    assert same.all()
