"""Autotuning keeps the automatic launch shapes where nothing it tries is faster (needs a GPU)."""
import numpy as np
import pytest

from leven_amd import mesher, workloads

pytestmark = pytest.mark.gpu


def _density_us(b):
    for _ in range(5):
        b.run_timed()
    return 1e3 * float(np.median([b.run_timed()["density"] for _ in range(31)]))


@pytest.mark.parametrize("chunks", [1, 2])
def test_autotune_keeps_the_density_split(chunks):
    """A few cave chunks are cut into up to 33 column segments by default, which no candidate
    of the autotuner matches (6 segments take twice the time)."""
    w = workloads.terrain_512()
    mesher.init(w["desc"], w["seed"], 0)
    mesher.clear_csg_ops()
    b = mesher.Batch(64, chunks)
    b.set_chunks(w["mins"][192:192 + chunks], w["sizes"][:chunks])
    b.run()
    before = [[a.tobytes() for a in b.get_mesh(i)] for i in range(chunks)]
    automatic = _density_us(b)
    shapes = b.autotune(3)
    tuned = _density_us(b)
    print(f"autotune: {chunks} chunks, density {automatic:.1f} us automatic, {tuned:.1f} us tuned, {shapes}", flush=True)
    b.run()
    assert [[a.tobytes() for a in b.get_mesh(i)] for i in range(chunks)] == before
    b.close()
    assert tuned <= 1.35 * automatic
