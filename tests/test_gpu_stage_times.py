"""Stage times of a batch: a stage that launches nothing takes no time (needs a GPU)."""
import pytest

from leven_amd import mesher, workloads

pytestmark = pytest.mark.gpu


def test_stages_without_a_launch_take_no_time():
    w = workloads.terrain_512()
    mesher.init(w["desc"], w["seed"], 0)
    mesher.clear_csg_ops()
    b = mesher.Batch(16, 2)
    b.set_chunks([(0, -64, 0), (64, -64, 0)], [64, 64])
    for _ in range(3):
        ms = b.run_timed()
    b.close()
    empty = {"voxel_rows", "scan_voxels", "voxel_compact"}
    assert len(ms) == mesher.NUM_STAGES and empty < set(ms)
    assert all(ms[k] == 0.0 for k in empty), ms
    assert all(ms[k] > 0.0 for k in set(ms) - empty), ms
