"""How many chunk slots a memory budget holds: a 64^3 slot of full capacities has always fitted
69,684,480 bytes, and the smaller ones the sizes below (needs a GPU)."""
import pytest

from leven_amd import mesher, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("voxels,edges,active,slot_bytes", [
    (64, 0, 0, 69684480), (64, 262144, 131072, 32560128), (64, 131072, 12000, 7937280), (32, 0, 0, 8956160),
    (16, 0, 0, 1186816), (8, 0, 0, 170496), (4, 0, 0, 30720)])
def test_slots_of_a_budget(voxels, edges, active, slot_bytes):
    w = workloads.terrain_512()
    mesher.init(w["desc"], w["seed"], 0)
    mesher.clear_csg_ops()
    s = mesher.Server(voxels, 20 * slot_bytes, 4, 1, edges, active)
    assert s.stats()["slots"] >= 20
    s.close()
