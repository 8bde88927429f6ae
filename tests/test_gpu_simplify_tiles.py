"""The simplifier's tiles at their edges, against the oracle bit for bit (needs a GPU):
vertices numbered at random, so that a tile's triangles lie in no window of vertices;
vertices of high degree, whose sides fit no register run; and numbers of triangles and
draws around a tile and its half."""
import numpy as np
import pytest

from leven_amd import abi, mesher, workloads

pytestmark = pytest.mark.gpu

OFF = np.zeros(4, np.float32)


def _grid(n, m, seed, order):
    """A wavy sheet of n x m vertices; `order` numbers them: rows, random, or fans (every
    eighth vertex of a row is the tip of a fan over its neighbours)."""
    rng = np.random.default_rng(seed)
    y, x = (a.ravel() for a in np.mgrid[0:n, 0:m])
    v = np.zeros(n * m, abi.VERTEX_DTYPE)
    f = v.view(np.float32).reshape(n * m, -1)
    z = 0.3 * np.sin(0.4 * x) + 0.2 * np.cos(0.3 * y) + 0.02 * rng.random(n * m)
    f[:, 0:3], f[:, 3] = np.stack([x, z, y], 1), 1.0
    g = np.stack([-0.12 * np.cos(0.4 * x), np.ones(n * m), 0.06 * np.sin(0.3 * y)], 1)
    f[:, 4:7] = g / np.linalg.norm(g, axis=1)[:, None]
    i = (np.arange(n - 1)[:, None] * m + np.arange(m - 1)).ravel()
    t = np.concatenate([np.stack([i, i + m, i + 1], 1), np.stack([i + 1, i + m, i + m + 1], 1)]).astype(np.int32)
    t = t.reshape(2, -1, 3).transpose(1, 0, 2).reshape(-1, 3)
    if order == "fans":  # bands of 2 x 24 strips meet in one vertex each
        tips = np.arange(0, n * m, 24) + 23
        tips = tips[tips < n * m]
        t = np.concatenate([[[a - k, a - k - 1, a] for k in range(1, 22)] for a in tips] * 2).astype(np.int32)
        t = np.concatenate([t, t[:, [1, 0, 2]]])
    if order == "random":
        to = rng.permutation(n * m).astype(np.int32)
        w = np.empty_like(v)
        w[to] = v
        v, t = w, to[t]
    return v, np.ascontiguousarray(t)


@pytest.mark.parametrize("n, m, order", [(23, 24, "rows"), (17, 33, "rows"), (90, 100, "rows"), (90, 100, "random"),
                                         (12, 96, "fans"), (40, 50, "random")])
def test_tiles_match_oracle(oracle, n, m, order):
    mesher.init(workloads.terrain_desc(), 2, 0)
    ctx = mesher.Context(64)
    v, t = _grid(n, m, n, order)
    for kw in (dict(max_error=1e9, max_edge_len=100.0, min_cos_angle=-1.0),
               dict(max_error=1e9, max_edge_len=100.0, min_cos_angle=-1.0, edge_fraction=1.0, max_iterations=25),
               dict(max_error=12.0, min_cos_angle=0.2)):
        opt = abi.simplify_options(256, **kw)
        print(f"simplify tiles: {n} x {m} {order} {kw}", flush=True)
        vo, to, so = oracle.simplify_mesh(v, t, OFF, opt)
        assert len(to) < len(t)
        vg, tg, sg = ctx.simplify_mesh(v, t, OFF, opt)
        assert vg.tobytes() == vo.tobytes() and tg.tobytes() == to.tobytes()
        assert sg == (int(so[0]), int(so[1]))
    ctx.close()
