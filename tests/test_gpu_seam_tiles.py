"""The two forms of the seam pass give the same bytes over the request sizes at which the
grid-wide form changes its launches: the lanes that make one seam's tile lists (64 for up
to 16 seams, fewer for more), tiles dealt over every XCD or kept to one (64 seams), and
small or large tiles (2^20 leaves in one request).

Seams are lists of made-up nodes, a band round a wavy surface and scattered ones, on the
faces of eight chunks.  tests/test_gpu_seams.py holds both forms against the oracle."""
import os

import numpy as np
import pytest

from leven_amd import mesher, workloads
from leven_amd.abi import SEAM_DTYPE

pytestmark = pytest.mark.gpu


def _lists(seed, scattered):
    rng = np.random.default_rng(seed)
    x, y, z = (a.ravel() for a in np.mgrid[0:64, 0:64, 0:64])
    face = np.zeros(x.shape, bool)
    for a in (x, y, z):
        face |= (a == 0) | (a == 63)
    x, y, z = x[face], y[face], z[face]
    out = []
    for k in range(8):
        o = np.array([k >> 2 & 1, k >> 1 & 1, k & 1])
        g = [v + 64 * s for v, s in zip((x, y, z), o)]
        band = np.abs(g[1] - 64 - 10 * np.sin(0.15 * g[0] + seed) - 8 * np.cos(0.2 * g[2])) <= 1.2
        at = np.flatnonzero(band | (rng.random(x.shape) < scattered))
        n = np.zeros(len(at), SEAM_DTYPE)
        words = n.view(np.int32).reshape(len(at), -1)
        words[:, :4] = np.stack([x[at], y[at], z[at], rng.integers(0, 1 << 16, len(at))], 1)
        n.view(np.float32).reshape(len(at), -1)[:, 4:] = rng.random((len(at), words.shape[1] - 4), np.float32)
        out.append(dict(min=tuple(256 * int(v) for v in o), size=256, neighbour=k, nodes=n))
    return out


@pytest.mark.parametrize("seams, scattered", [(1, 0.0), (1, 0.5), (17, 0.01), (63, 0.01), (64, 0.01), (300, 0.05)])
def test_forms_agree(seams, scattered):
    mesher.init(workloads.terrain_desc(), 2, 0)
    ctx = mesher.Context(64)
    kinds = [_lists(k, scattered) for k in range(min(seams, 3))]
    hosts = [((0, 0, 0), 256, (1.0, 0.5, 0.25))] * seams
    sources = [kinds[i % len(kinds)] for i in range(seams)]
    offered = sum(len(q["nodes"]) for q in kinds[0])
    got = {}
    old = os.environ.get("LVN_SEAM_PATH")
    try:
        for path in ("grid", "workgroup"):
            os.environ["LVN_SEAM_PATH"] = path
            got[path] = ctx.seam_meshes(hosts, sources, [offered + 4096] * seams, [4 * offered + 4096] * seams)
    finally:
        if old is None:
            del os.environ["LVN_SEAM_PATH"]
        else:
            os.environ["LVN_SEAM_PATH"] = old
        ctx.close()
    assert sum(len(t) for _, t in got["grid"]) > 0
    for (v, t), (w, u) in zip(got["grid"], got["workgroup"]):
        assert v.tobytes() == w.tobytes() and t.tobytes() == u.tobytes()
