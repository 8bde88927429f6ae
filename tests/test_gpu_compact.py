"""Edge and voxel lists in both of their walks (a lane per list entry where rows are sparse,
a lane per position where they are dense) and both launch forms (four waves per 64 rows for
a few chunks, one for many): one chunk's lists against the oracle's, and meshes of a batch
of 64, whose density pass stores solid planes in y-segments, against that chunk's (needs a
GPU)."""
import numpy as np
import pytest

from leven_amd import abi, mesher, workloads
from oracle import py_oracle

pytestmark = pytest.mark.gpu

FIELDS = {
    # a plane: 64 y-edges and one at x = 64 in each of a few rows
    "plane": (abi.field_desc(height_octaves=0), 2, 0),
    # under the ground, where most rows hold many edges
    "caves": (workloads.terrain_desc(), 2, -2048),
    # a few edges a row
    "hills": (workloads.heightfield_desc(), 1, -128),
    "leven": (workloads.leven_desc(), workloads.LEVEN_SEED, 2320),
}


@pytest.mark.parametrize("field", FIELDS)
@pytest.mark.parametrize("voxels", [4, 32, 64])
def test_lists_match_oracle(field, voxels):
    desc, seed, y = FIELDS[field]
    mesher.init(desc, seed, 0)
    mesher.clear_csg_ops()
    size = 4 * voxels
    mn = (64, y // size * size if abs(y) > 1000 else -2 * voxels, 128)
    print(f"compact: {field} N={voxels}", flush=True)
    ctx = mesher.Context(voxels)
    g = ctx.debug_stages(mn, size)
    c = py_oracle.Chunk(voxels).generate(desc, py_oracle.perm_table(seed), mn, size).build()
    ids, data = c.edges()
    assert (g["edge_ids"] == ids).all() and len(g["edge_ids"]) == len(ids)
    assert np.ascontiguousarray(g["edge_data"], np.float32).tobytes() == np.ascontiguousarray(data, np.float32).tobytes()
    assert (g["voxel_codes"] == c.voxels()[0]).all()
    want = ctx.generate_chunk_mesh(mn, size)
    n = 64
    b = mesher.Batch(voxels, n)
    b.set_chunks([mn] * n, [size] * n)
    for ysplit in (0, 1, 5, voxels):  # y-segments of the planes, the last ones short or empty
        b.set_tuning(density_ysplit=ysplit)
        b.run()
        assert b.counts()[:n, 4].max() == 0
        for i in (0, 1, n // 2, n - 1):
            for got, ref in zip(b.get_mesh(i), want):
                assert got.shape == ref.shape and got.tobytes() == ref.tobytes()
    b.close()
    ctx.close()
