"""Chunks that are all solid or all air, which the batch's bookkeeping kernels pass by, in
slots that held a surface before and hold one again after; brushes in such chunks; and the
line heights over them.  Every mesh equals the one-chunk context's (needs a GPU)."""
import numpy as np
import pytest

from leven_amd import mesher, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxels", [4, 16, 64])
@pytest.mark.parametrize("field", ["height", "caves"])
def test_uniform_chunks_in_reused_slots(voxels, field):
    desc = workloads.heightfield_desc() if field == "height" else workloads.terrain_desc()
    mesher.init(desc, 3, 0)
    mesher.clear_csg_ops()
    size = 4 * voxels
    far = 64 * size + 256  # beyond the height term's amplitude
    surface, sky, rock = [(0, -size, 0), (size, 0, 0), (0, 0, size)], (0, far, 0), (0, -far // size * size, 0)
    hole = (4 * size, far, 0)  # a sky chunk with a brush in it
    op = workloads.make_ops(1, seed=1, spheres=1)[0]
    op["type"], op["material"] = 0, 2
    op["origin"][0, :3] = [hole[0] / 4 + voxels / 2, hole[1] / 4 + voxels / 2, hole[2] / 4 + voxels / 2]
    op["dims"][0, :3] = 0.3 * voxels
    mesher.store_csg_op(op[0], hole, [hole[0] + size, hole[1] + size, hole[2] + size])
    b = mesher.Batch(voxels, 4)
    ctx = mesher.Context(voxels)
    for chunks in (surface + [sky], [sky, rock, hole, surface[0]], [rock, surface[1], sky, hole],
                   [sky, sky, rock, sky], surface[::-1] + [hole]):
        for lines in (1, 2):
            b.set_chunks(chunks, [size] * 4)
            b.set_tuning(height_lines=lines)
            b.run()
            k = b.counts().copy()
            for i, mn in enumerate(chunks):
                print(f"uniform chunks: N={voxels} {field} {mn} in slot {i}", flush=True)
                ctx.free_chunk(mn, size)
                want = ctx.generate_chunk_mesh(mn, size)
                for got, ref in zip(b.get_mesh(i), want):
                    assert got.shape == ref.shape and got.tobytes() == ref.tobytes()
                if mn == sky:
                    assert (k[i] == 0).all()
    mesher.clear_csg_ops()
    b.close()
    ctx.close()
