"""Batch and server meshes read into pinned host memory (one launch) equal those read into
ordinary memory, at every alignment the C ABI allows, with some outputs left out, after a
run, a second run over other chunks and a simplification (needs a GPU)."""
import ctypes as C

import numpy as np
import pytest

from leven_amd import abi, mesher, workloads

pytestmark = pytest.mark.gpu


class Pinned:
    def __init__(self, nbytes):
        mesher.lib()
        self.hip = C.CDLL("libamdhip64.so.7")
        self.hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        self.hip.hipHostFree.argtypes = [C.c_void_p]
        self.p = C.c_void_p()
        assert self.hip.hipHostMalloc(C.byref(self.p), nbytes, 0) == 0
        self.bytes = np.ctypeslib.as_array(C.cast(self.p, C.POINTER(C.c_uint8)), (nbytes,))

    def free(self):
        self.hip.hipHostFree(self.p)


def _read(get, mem, offsets, mesh, skip=None):
    """The mesh read at `offsets` bytes into mem's three thirds; nothing outside it is written."""
    third = len(mem.bytes) // 3 // 16 * 16
    mem.bytes[:] = 0xA5
    out = [None if k == skip else mem.p.value + k * third + offsets[k] for k in range(3)]
    n = [C.c_int32() for _ in range(3)]
    cap = 1 << 24
    assert get(out[0], cap, C.byref(n[0]), out[1], cap, C.byref(n[1]), out[2], cap, C.byref(n[2])) == abi.LVN_OK
    for k, want in enumerate(mesh):
        assert n[k].value == len(want)
        got = mem.bytes[k * third:(k + 1) * third]
        raw = want.tobytes() if k != skip else b""
        assert got[offsets[k]:offsets[k] + len(raw)].tobytes() == raw, (k, offsets)
        assert (got[:offsets[k]] == 0xA5).all() and (got[offsets[k] + len(raw):] == 0xA5).all(), (k, offsets)


@pytest.mark.parametrize("voxels", [4, 16, 64])
def test_pinned_reads_equal_ordinary_ones(voxels):
    w = workloads.terrain_512()
    mesher.init(w["desc"], w["seed"], 0)
    mesher.clear_csg_ops()
    size = 4 * voxels
    mem = Pinned(24 << 20)
    b = mesher.Batch(voxels, 3)
    server = mesher.Server(voxels, 1 << 30, 4, 1, 0, 0)
    L = mesher.lib()
    try:
        for step, x in (("run", 0), ("other chunks", 5), ("simplified", 5)):
            mins = [(x * size, -size, 0), (x * size, 40 * size, 0), (x * size, 0, size)]  # the second is sky
            if step == "simplified":
                b.simplify(abi.simplify_options_per_voxel(max_error=50.0, min_cos_angle=-1.0))
            else:
                b.set_chunks(mins, [size] * 3)
                b.run()
            for i in range(3):
                mesh = b.get_mesh(i)
                for offsets in ((0, 0, 0), (16, 8, 16), (4, 4, 4), (8, 12, 24)):
                    print(f"readback: N={voxels} {step} chunk {i} at {offsets}", flush=True)
                    _read(lambda *a: L.lvn_batch_get_mesh(b._h, i, *a), mem, offsets, mesh)
                for skip in range(3):
                    _read(lambda *a: L.lvn_batch_get_mesh(b._h, i, *a), mem, (0, 4, 0), mesh, skip)
            if step != "simplified":
                tickets = server.submit_meshes(mins, [size] * 3)
                server.drain()
                for i, t in enumerate(tickets):
                    _read(lambda *a: L.lvn_server_get_mesh(server._h, int(t), *a), mem, (0, 4, 16), b.get_mesh(i))
    finally:
        b.close()
        server.close()
        mem.free()
