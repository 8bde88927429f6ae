"""Batches in which many chunks lie under brushes, each under its own number of them (round the
wave's size and the kernels' dispatch lines), against the oracle bit for bit: more lists than a
wave has lanes, lists longer than a wave, chunks with and without edges between them (needs a GPU)."""
import numpy as np
import pytest

from leven_amd import mesher, workloads
from oracle import py_oracle

pytestmark = pytest.mark.gpu


def _ops(n, seed, mn, voxels, scale):
    """n brushes over the chunk at mn, some the same, nearly flat, huge or inside out."""
    rng = np.random.default_rng(seed)
    half = 0.5 * voxels * scale
    ops, _ = workloads.make_ops(n, seed=seed, rotated=True, extent=voxels * scale, y_range=(-half, half),
                                size_range=(0.5 * scale, 0.25 * voxels * scale))
    for k in range(0, n, 5):
        ops[k] = ops[rng.integers(0, n)]  # every sample ties
    for k in range(1, n, 7):
        ops[k]["dims"][rng.integers(0, 3)] = 0.01
    if n > 25:
        ops[n // 3]["dims"][:3] = 3.0 * voxels * scale  # holds the whole chunk
        ops[n // 4]["dims"][:3] = -1.0                   # holds nothing
    for op in ops:
        op["origin"][0] += mn[0] / 4
        op["origin"][1] += mn[1] / 4 + half
        op["origin"][2] += mn[2] / 4
    return ops


def _check(desc, voxels, mins, size, counts, seed):
    scale = size // (4 * voxels)
    mesher.init(desc, 2, 0)
    mesher.clear_csg_ops()
    lists = []
    for k, (mn, n) in enumerate(zip(mins, counts)):
        ops = _ops(n, seed + k, mn, voxels, scale) if n else np.zeros(0, workloads.CSG_OP_DTYPE)
        for op in ops:
            mesher.store_csg_op(op, mn, [v + size for v in mn])
        lists.append(ops)
    b = mesher.Batch(voxels, len(mins))
    b.set_chunks(mins, [size] * len(mins))
    perm = py_oracle.perm_table(2)
    try:
        for step in range(2):  # the second run replays the captured graph
            b.run()
            meshed = 0
            for k, mn in enumerate(mins):
                c = py_oracle.Chunk(voxels).generate(desc, perm, mn, size, ops=lists[k]).build()
                v, t, s = b.get_mesh(k)
                where = f"chunk {k} of {len(mins)}, {len(lists[k])} ops, run {step}"
                want = c.vertices() if len(c.triangles()) else c.vertices()[:0]
                assert len(t) == len(c.triangles()) and (t == c.triangles()).all(), where
                assert v.tobytes() == want.tobytes(), where
                assert s.tobytes() == c.seams().tobytes(), where
                meshed += len(t) > 0
            assert meshed >= sum(n > 0 for n in counts) // 2
    finally:
        mesher.clear_csg_ops()
        b.close()


@pytest.mark.parametrize("voxels,lod,counts", [
    (16, 0, [19]), (16, 0, [20]), (32, 1, [20, 0, 19]), (16, 0, [65, 0, 40, 0, 0, 0, 0, 1]),
    (16, 0, [65, 0, 40, 0, 0, 0, 0, 1, 0]), (64, 0, [300] + [0] * 8), (16, 1, [1, 19, 20, 40, 63, 64, 65, 130, 300, 0, 2]),
    (4, 0, [3, 65, 0] * 30)])
def test_brushed_batches_match_oracle(voxels, lod, counts):
    size = 4 * voxels << lod
    mins = [(40 * size * k, -size // 2 // 4 * 4, 8 * size * (k % 3)) for k in range(len(counts))]
    print(f"brush lists: N={voxels} lod={lod} {counts[:12]}", flush=True)
    _check(workloads.heightfield_desc(), voxels, mins, size, counts, 11 * len(counts) + voxels)


def test_more_lists_than_lanes():
    """150 chunks, 100 of them brushed, some high in the air with and without a brush's surface."""
    rng = np.random.default_rng(5)
    counts = [int(rng.choice([0, 1, 2, 5, 20, 66])) if k % 3 else 0 for k in range(150)]
    size = 64
    mins = [(40 * size * (k % 25), (-size // 2 if k % 4 else 30 * size), 40 * size * (k // 25)) for k in range(150)]
    print(f"brush lists: {sum(c > 0 for c in counts)} of {len(counts)} chunks", flush=True)
    _check(workloads.terrain_desc(), 16, mins, size, counts, 900)


def _stage_us(chunks, stage):
    """The stage's time for that many 4^3 chunks under a brush each."""
    mesher.init(workloads.heightfield_desc(), 2, 0)
    mesher.clear_csg_ops()
    mins = [(40 * 16 * (k % 64), -8, 40 * 16 * (k // 64)) for k in range(chunks)]
    for k, mn in enumerate(mins):
        mesher.store_csg_op(_ops(1, k, mn, 4, 1)[0], mn, [v + 16 for v in mn])
    b = mesher.Batch(4, chunks)
    b.set_chunks(mins, [16] * chunks)
    for _ in range(5):
        b.run_timed()
    us = 1e3 * float(np.median([b.run_timed()[stage] for _ in range(21)]))
    mesher.clear_csg_ops()
    b.close()
    return us


@pytest.mark.parametrize("stage", ["csg", "edge_cross"])
def test_a_wave_reads_only_its_own_chunks(stage):
    """Twenty times the brushed chunks, all but empty: a pass whose waves each went through the
    whole list of them would take twenty times as long."""
    few, many = _stage_us(60, stage), _stage_us(1200, stage)
    print(f"brush lists: {stage} {few:.1f} us for 60 chunks, {many:.1f} us for 1,200", flush=True)
    assert many <= 6 * few
