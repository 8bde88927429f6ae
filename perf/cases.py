"""What this mesher is measured on: the calls its users make, over their real range of sizes.

A case names a form (which entry points a pass goes through), a field (what the world is
made of) and sizes.  The worlds are this repository's own: the six-octave heightfield, the
heightfield with caves and its brushes, and the reference's terrain field.  The seed of a
case's inputs moves the place in the world (and the camera) that is meshed, so another
seed is other chunks; the world itself is entered once, as a program does.
"""
import ctypes as C
import math

import numpy as np
import torch

from leven_amd import abi, mesher, workloads

CHUNK = workloads.CHUNK_SIZE
R = workloads.LOD_MAX_NODE_SIZE


def listed():
    return [
        # the smallest call: one 16^3 chunk of a heightfield through the drop-in context, mesh on the host
        dict(name="dropin_16_height", form="chunk", field="height", brushes=0, voxels=16, lod=0),
        # the drop-in call as the application makes it: one fresh 64^3 chunk with caves
        dict(name="dropin_64_caves", form="chunk", field="caves", brushes=0, voxels=64, lod=0),
        # one chunk under stored brushes without allocation, outputs in device memory (a render loop)
        dict(name="scratch_64_leven", form="scratch", field="leven", brushes=256, voxels=64, lod=0, flags=0),
        # a player's edit: a brush filled in, the chunk re-meshed, dug out again, re-meshed
        dict(name="edit_64_caves", form="edit", field="caves", brushes=0, voxels=64, lod=0, ops=4),
        # a camera step: the 24 chunks nearest the camera staged, meshed and fetched to the host
        dict(name="step_24_leven", form="batch", field="leven", brushes=256, voxels=64, near=24, flags=0),
        # the precision form: a 4^3 block under rotated boxes, compensated QEF, fetched to the host
        dict(name="precise_64_boxes", form="batch", field="caves", brushes=1024, voxels=64, bx=4, by=4, bz=4, lod=0,
             flags=abi.CTX_PRECISE_QEF),
        # the 6-LOD clipmap, 1,800 chunks, over the reference's terrain, with the 16 nearest seams, left in HBM
        dict(name="clipmap_leven", form="resident", field="leven", brushes=256, voxels=64, near=1800, hosts=16),
        # the 8x8x8 region of caves with its 256 brushes and all its seams, seams read back
        dict(name="region_512_caves", form="region", field="caves", brushes=256, voxels=64, bx=8, by=8, bz=8, lod=0),
        # coarse underground tiles, where nearly every voxel is active, and their seams, left in HBM
        dict(name="far_50_caves", form="resident", field="caves", brushes=0, voxels=64, bx=5, by=2, bz=5, lod=5,
             hosts=16),
        # meshing plus simplification of a block, the simplified meshes fetched to the host
        dict(name="simplify_64_caves", form="simplify", field="caves", brushes=0, voxels=64, bx=4, by=4, bz=4, lod=0),
        # one seam of the drop-in form: host lists in, host mesh out
        dict(name="stitch_1_caves", form="stitch", field="caves", brushes=0, voxels=64, lod=1),
        # the server under a moving camera: two bursts that evict each other's chunks, meshes fetched
        dict(name="serve_48_caves", form="serve", field="caves", brushes=256, voxels=64, near=48, lanes=3),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    form = rng.choice(["chunk", "scratch", "edit", "batch", "batch", "resident", "resident", "region", "simplify",
                       "stitch", "serve"])
    field = rng.choice(["height", "caves", "leven"])
    brushes = rng.choice([0, 0, rng.randint(3, 400)])
    c = dict(form=form, field=field, brushes=brushes, voxels=64)
    if form in ("chunk", "scratch"):
        if form == "chunk":  # a context keeps a brushed chunk's field, and its next mesh would start from that
            c["brushes"] = 0
        c.update(voxels=rng.choice([4, 8, 16, 32, 64, 64, 64]), lod=rng.randint(0, 5))
        if form == "scratch":  # its fixed area holds 65,536 active voxels
            c.update(lod=rng.randint(0, 1) if field == "caves" else c["lod"],
                     flags=rng.choice([0, 0, abi.CTX_PRECISE_QEF, abi.CTX_FP16_DENSITY]))
    elif form == "edit":
        c.update(brushes=0, voxels=rng.choice([16, 32, 64, 64]), lod=rng.randint(0, 2), ops=rng.randint(1, 12))
    elif form == "batch":
        c.update(near=_log_int(rng, 2, 120 if field == "caves" else 300), flags=rng.choice([0, 0, abi.CTX_PRECISE_QEF, abi.CTX_FP16_DENSITY]))
    elif form == "resident":
        if field == "caves":
            bx, bz, lod = rng.randint(2, 5), rng.randint(2, 5), rng.randint(0, 5)
            c.update(bx=bx, by=2, bz=bz, lod=lod, hosts=rng.randint(1, (bx - 1) * (bz - 1)))
        else:
            c.update(near=_log_int(rng, 40, 1700), hosts=rng.randint(4, 16))
    elif form in ("region", "simplify"):
        top = 6 if form == "region" else 4
        c.update(bx=rng.randint(2, top), by=rng.randint(2, 4), bz=rng.randint(2, top), lod=rng.randint(0, 2))
    elif form == "stitch":
        c.update(lod=rng.randint(0, 3), brushes=0)
    else:
        c.update(near=_log_int(rng, 6, 60), lanes=rng.randint(1, 3))
    return c


# ---------------------------------------------------------------- worlds and places

NOISE_SEED = {"height": 1, "caves": 2, "leven": workloads.LEVEN_SEED}
_world = None


def _enter(case):
    """The case's world: field, noise seed and its history of stored brushes, set once."""
    global _world
    key = (case["field"], case["brushes"])
    if _world == key:
        return
    desc = {"height": workloads.heightfield_desc, "caves": workloads.terrain_desc,
            "leven": workloads.leven_desc}[case["field"]]()
    mesher.init(desc, NOISE_SEED[case["field"]], 0)
    mesher.clear_csg_ops()
    n = case["brushes"]
    if n > 512:  # the precision workload's rotated boxes
        ops, aabbs = workloads.make_ops(n, seed=3, spheres=0, rotated=True)
    elif case["field"] == "leven" and n:
        w = workloads.clipmap_leven()
        ops, aabbs = [np.concatenate([w[k], w[k]])[:n] for k in ("ops", "aabbs")]
    else:
        ops, aabbs = workloads.make_ops(n, seed=2)
    for op, bb in zip(ops, aabbs):
        mesher.store_csg_op(op, bb[:3], bb[3:])
    _world = key


def _count(case, mins, sizes):
    """Edges, voxels, triangles, seam nodes, status and re-solves of each chunk."""
    b = mesher.Batch(case["voxels"], len(sizes))
    b.set_chunks(mins, sizes)
    b.run()
    k = b.counts().copy()
    b.close()
    return k


def _column(case, seed, size):
    """The chunk with most surface in a column of the world that the seed picks."""
    x, z = (seed * 37) % 29 - 14, (seed * 17) % 31 - 15
    if case["brushes"]:  # the brushes lie over [0, 512) voxels, leven's around its camera
        x, z = (seed * 37) % 8, (seed * 5) % 7
        if case["field"] == "leven":
            x = int(workloads.LEVEN_CAMERA[0]) // size + seed % 3 - 1
            z = int(workloads.LEVEN_CAMERA[2]) // size + seed // 3 % 3 - 1
    reach = max(2 * size, 128)
    ys = range(0, max(6144, size), size) if case["field"] == "leven" else range(-reach, reach, size)
    mins = np.array([[x * size, y, z * size] for y in ys], np.int32)
    k = _count(case, mins, np.full(len(mins), size, np.int32))
    return tuple(int(v) for v in mins[int(np.argmax(k[:, 1]))])


def _size(case):
    return 4 * case["voxels"] << case["lod"]


def _camera(case, seed):
    if case["field"] == "leven":
        if not case["brushes"]:
            x, y, z = _column(case, seed, CHUNK)
            return np.array([x + 100.0, y + 192.0, z + 60.0])
        cx, _, cz = workloads.LEVEN_CAMERA
        dx, dz = ((seed * 37) % 17 - 8) * 24.0, ((seed * 11) % 13 - 6) * 32.0
        h0, sx, sz = workloads.LEVEN_SURFACE
        return np.array([cx + dx, 4.0 * (h0 + 16.0) + sx * dx + sz * dz, cz + dz])
    return np.array([((seed * 37) % 41) * 49.0 + 7.0, (seed * 13) % 9 * 16.0 - 64.0, ((seed * 11) % 43) * 47.0 + 3.0])


def _place(case, seed):
    """Chunk mins and sizes of a batch: the nearest of the clipmap's selection around a
    camera, or a block of chunks of one voxel size across the surface."""
    if "near" in case:
        cam = _camera(case, seed)
        cm = mesher.Clipmap((-14 * R, -R, -14 * R), (14 * R, R, 14 * R))
        mins, sizes = cm.update(cam)["selected"]
        cm.close()
        d = np.maximum(np.maximum(mins - cam, 0.0), cam - (mins + sizes[:, None]))
        order = np.argsort((d * d).sum(axis=1), kind="stable")[: case["near"]]
        return mins[order].copy(), sizes[order].copy()
    size = _size(case)
    ox, oz = (seed * 7) % 9 - 4, (seed * 5) % 11 - 5
    if case["brushes"]:
        ox, oz = (seed * 7) % 5 - 2, (seed * 5) % 3 - 1
    oy = -(case["by"] // 2)
    if case["field"] == "leven":
        ox, above, oz = [v // size for v in _column(case, seed, size)]
        oy += above
    mins = np.array([[(x + ox) * size, (y + oy) * size, (z + oz) * size] for z in range(case["bz"])
                     for y in range(case["by"]) for x in range(case["bx"])], np.int32)
    return mins, np.full(len(mins), size, np.int32)


# ---------------------------------------------------------------- states

class _State:
    pass


def _caps(case):
    """Per-chunk capacities as a program sets them: a surface without caves keeps a 64^3 chunk
    under 32,768 active voxels, fine caves under 131,072; coarse caves need the full ones."""
    if case["field"] != "caves" and case.get("near", 0) > 400:
        return 65536, 32768
    return (262144, 131072) if case.get("lod", 0) == 0 and "near" not in case else (0, 0)


def _rows(case, chunks):
    """Room for the meshes of so many chunks: vertices, triangles, seam nodes.  A program's
    buffers have fixed sizes (the application's own are); the counts say how much is filled."""
    n3 = case["voxels"] ** 3
    if case["field"] != "caves":
        one, each = 32768, 8192
    elif "near" in case:
        one, each = 65536, 24576 if chunks <= 60 else 40960
    else:
        one, each = (65536, 24576) if case["lod"] == 0 else (131072, 32768) if case["lod"] <= 2 else (262144, 98304)
    v = min(n3, one) + chunks * min(n3, each)
    return v, 5 * v // 2, v // 4 + min(n3, 24576)


def _buffers(s, rows, **kw):
    v, t, q = rows
    s.v, s.t, s.q = [torch.zeros((r, w), dtype=d, **kw) for r, w, d in
                     ((v, 12, torch.float32), (t, 3, torch.int32), (q, 12, torch.int32))]
    s.caps = rows


def _meshes(s, got):
    """The buffers, and how many vertices, triangles and seam nodes they hold."""
    return dict(vertices=s.v, triangles=s.t, seam_voxels=s.q[:, :4], seam_points=s.q.view(torch.float32)[:, 4:],
                filled=np.array(got, np.int32))


def _batch(case, seed):
    s = _State()
    s.mins, s.sizes = _place(case, seed)
    s.b = mesher.Batch(case["voxels"], len(s.sizes), *_caps(case), case.get("flags", 0))
    s.b.set_chunks(s.mins, s.sizes)
    s.b.run()
    s.k = s.b.counts().copy()
    return s


def _grid_seams(case, s):
    """Host nodes of a block with all seven upper neighbours, and the lists each one gathers."""
    at = {tuple(int(v) for v in m): i for i, m in enumerate(s.mins)}
    size = int(s.sizes[0])
    hosts, lists = [], []
    for m in at:
        around = [tuple(m[a] + size * o[a] for a in range(3)) for o in workloads.CHILD_MIN_OFFSETS]
        if all(p in at for p in around):
            hosts.append((m, size, (1.0, 1.0, 1.0)))
            lists.append([dict(min=p, size=size, neighbour=i, nodes=None) for i, p in enumerate(around)
                          if s.k[at[p], 3] > 0])
    n = case.get("hosts", len(hosts))
    return hosts[:n], lists[:n]


def _clipmap_seams(case, s, seed):
    """The seams the request producer asks for once the selection is meshed: the nearest ones."""
    cm = mesher.Clipmap((-14 * R, -R, -14 * R), (14 * R, R, 14 * R))
    mins, sizes = cm.update(_camera(case, seed))["to_mesh"]
    meshed = {(*map(int, m), int(z)): k for m, z, k in zip(s.mins, s.sizes, s.k)}
    zero = np.zeros(6, np.int32)
    got = [meshed.get((*map(int, m), int(z)), zero) for m, z in zip(mins, sizes)]
    reqs, srcs, n, _ = cm.commit([(k[4], k[2], k[3]) for k in got])
    cm.close()
    rank = {key: i for i, key in enumerate(meshed)}
    near = sorted(range(n), key=lambda i: rank.get((*reqs[i].host_min, reqs[i].host_size), 1 << 30))[: case["hosts"]]
    hosts, lists = [], []
    for i in near:
        q = reqs[i]
        hosts.append((tuple(q.host_min), q.host_size, tuple(q.colour)[:3]))
        lists.append([dict(min=tuple(x.min), size=x.size, neighbour=x.neighbour, nodes=None)
                      for x in srcs[q.first_source: q.first_source + q.n_sources]])
    return hosts, lists


def _seam_call(s, hosts, lists):
    """The C call's arguments, which a program keeps while its selection stands."""
    flat, s.reqs = [], (abi.SeamReq * max(1, len(hosts)))()
    for q, (mn, size, colour), l in zip(s.reqs, hosts, lists):
        q.host_min[:], q.host_size, q.colour[:] = mn, size, [*colour, 0.0]
        q.first_source, q.n_sources = len(flat), len(l)
        flat += l
    s.hosts, s.srcs, s.outs = len(hosts), abi.seam_sources(flat), (abi.SeamOut * max(1, len(hosts)))()


def _stitch(s):
    mesher.check(mesher.lib().lvn_batch_seam_meshes(s.b._h, s.hosts, C.cast(s.reqs, C.c_void_p),
                                                    C.cast(s.srcs, C.c_void_p), C.cast(s.outs, C.c_void_p)), "seams")


def _seam_rows(case):
    """Room for the seams of a case: a seam holds about as many nodes as its chunks' faces."""
    hosts = case.get("hosts", 1)
    if case["form"] == "region":
        hosts = (case["bx"] - 1) * (case["by"] - 1) * (case["bz"] - 1)
    per = 8192 if case["field"] != "caves" else 16384 if case.get("lod", 0) == 0 else 98304
    v = 16384 + hosts * per
    return v, 3 * v, 1


class _Device:
    """Device memory of the library as an array that torch can read."""

    def __init__(self, p, n, kind):
        self.__cuda_array_interface__ = dict(data=(p, False), shape=(n,), typestr=kind, version=3)


def prepare(case, seed):
    _enter(case)
    form, n = case["form"], case["voxels"]
    if form in ("batch", "simplify"):
        s = _batch(case, seed)
        _buffers(s, _rows(case, len(s.sizes)), pin_memory=True)
    elif form in ("resident", "region"):
        s = _batch(case, seed)
        hosts, lists = _grid_seams(case, s) if "bx" in case else _clipmap_seams(case, s, seed)
        _seam_call(s, hosts, lists)
        if form == "region":  # each seam's place in the buffers, of the size that the first answer names
            _buffers(s, _seam_rows(case), pin_memory=True)
            _stitch(s)
            at = [0, 0]
            for o in s.outs[: s.hosts]:
                o.v, o.v_cap = s.v.data_ptr() + 48 * at[0], o.nv
                o.tri, o.tri_cap = s.t.data_ptr() + 12 * at[1], o.nt
                at = [at[0] + o.nv, at[1] + o.nt]
            assert at[0] <= s.caps[0] and at[1] <= s.caps[1]
        else:
            _buffers(s, _seam_rows(case), device="cuda")
    elif form == "stitch":
        s = _State()
        x, y, z = _column(case, seed, _size(case))
        s.min, s.size = np.array([x, y, z], np.int32), _size(case)
        around = [tuple(int(v) for v in np.add((x, y, z), np.multiply(o, _size(case))))
                  for o in workloads.CHILD_MIN_OFFSETS]
        b = mesher.Batch(n, 8)
        b.set_chunks(around, [_size(case)] * 8)
        b.run()
        k = b.counts().copy()
        s.nodes = [dict(min=p, size=_size(case), neighbour=i, nodes=b.get_seam_nodes(i, k))
                   for i, p in enumerate(around) if k[i, 3]]
        b.close()
        s.srcs = abi.seam_sources(s.nodes)
        s.colour = np.array([1.0, 1.0, 1.0], np.float32)
        s.ctx = mesher.Context(n)
        _buffers(s, _seam_rows(case))
    elif form == "serve":
        s = _State()
        mins, sizes = _place(dict(case, near=2 * case["near"]), seed)
        half = len(sizes) // 2
        s.lists = [(mins[i::2][:half], sizes[i::2][:half]) for i in (0, 1)]
        _buffers(s, _rows(case, 2 * half), pin_memory=True)
        probe = mesher.Server(n, 1 << 30, 8, 1, 0, 0)  # slots of a budget: the bytes of one
        slot = (1 << 30) // max(1, probe.stats()["slots"])
        probe.close()
        s.server = mesher.Server(n, slot * half, -(-half // case["lanes"]), case["lanes"], 0, 0)
    else:
        s = _State()
        s.size = _size(case)
        s.min = np.array(_column(case, seed, s.size), np.int32)
        if form == "scratch":
            s.n, s.flags = n, case["flags"]
            _buffers(s, _rows(case, 1), device="cuda")
        else:
            s.ctx = mesher.Context(n)
            _buffers(s, _rows(case, 1))
        if form == "edit":
            s.other = _State()
            _buffers(s.other, s.caps)
            rng = np.random.default_rng(seed)
            scale = s.size // (4 * n)
            s.fill = np.zeros(case["ops"], abi.CSG_OP_DTYPE)
            for op in s.fill:
                op["brush"], op["material"] = rng.integers(0, 2), rng.integers(1, 4)
                op["origin"][:3] = s.min / 4 + rng.uniform(0.2, 0.8, 3) * n * scale + 0.5
                op["dims"][:3] = rng.uniform(0.03, 0.18) * n * scale
            s.dig = s.fill.copy()
            s.dig["type"], s.dig["material"] = 1, abi.MATERIAL_AIR
            _edit(s)  # the field is kept and the place has been dug once
    s.case = case
    return s


# ---------------------------------------------------------------- passes

class _Mesh:
    """The C calls' mesh arguments: where the next mesh goes in the buffers, and what came."""

    def __init__(self, s):
        self.p = (s.v.data_ptr(), s.t.data_ptr(), s.q.data_ptr())
        self.caps, self.at = s.caps, [0, 0, 0]
        self.got = C.c_int32(), C.c_int32(), C.c_int32()

    def call(self, fn, *args):
        (v, t, q), (a, b, c), at, (x, y, z) = self.p, self.caps, self.at, self.got
        mesher.check(fn(*args, v + 48 * at[0], a - at[0], C.byref(x), t + 12 * at[1], b - at[1], C.byref(y),
                        q + 48 * at[2], c - at[2], C.byref(z)), "mesh")
        self.at = [at[0] + x.value, at[1] + y.value, at[2] + z.value]


def _fetch(s, k):
    """Every mesh of the batch into the program's buffers, back to back."""
    m, get = _Mesh(s), mesher.lib().lvn_batch_get_mesh
    for i in np.flatnonzero(k[:, 0]):
        m.call(get, s.b._h, int(i))
    return _meshes(s, m.at)


def _generate(s, into):
    m = _Mesh(into)
    s.ctx.free_chunk(s.min, s.size)
    m.call(mesher.lib().lvn_generate_chunk_mesh, s.ctx._h, abi.vptr(s.min), s.size)
    return _meshes(into, m.at)


def _edit(s):
    s.ctx.apply_csg(s.fill, s.min, s.size)
    filled = _generate(s, s)
    s.ctx.apply_csg(s.dig, s.min, s.size)
    return filled, _generate(s, s.other)


def _resident_seams(s):
    """The seam meshes, which lie in device memory, into the program's own device buffers."""
    at = [0, 0]
    for i in range(s.hosts):
        v, t, nv, nt = s.b.seam_device_mesh(i)
        if nv:
            s.v[at[0]: at[0] + nv].view(-1).copy_(torch.as_tensor(_Device(v, 12 * nv, "<f4"), device="cuda"))
        if nt:
            s.t[at[1]: at[1] + nt].view(-1).copy_(torch.as_tensor(_Device(t, 3 * nt, "<i4"), device="cuda"))
        at = [at[0] + nv, at[1] + nt]
    torch.cuda.current_stream().synchronize()  # the library's next seams go to the same memory
    return dict(vertices=s.v, triangles=s.t, filled=np.array(at, np.int32))


def run(s):
    form = s.case["form"]
    if form == "chunk":
        return _generate(s, s)
    if form == "scratch":
        m = _Mesh(s)
        m.call(mesher.lib().lvn_generate_chunk_mesh_noalloc, s.n, s.flags, abi.vptr(s.min), s.size)
        return _meshes(s, m.at)
    if form == "edit":
        return _edit(s)
    if form == "batch":
        s.b.set_chunks(s.mins, s.sizes)
        s.b.run()
        k = s.b.counts()
        return dict(_fetch(s, k), counts=k)
    if form == "simplify":
        s.b.run()
        k = s.b.simplify(abi.simplify_options_per_voxel())
        return dict(_fetch(s, s.k), counts=k)
    if form in ("resident", "region"):
        s.b.run()
        k = s.b.counts()
        _stitch(s)
        if form == "resident":
            return dict(_resident_seams(s), counts=k)
        return dict(vertices=s.v, triangles=s.t, counts=k, sizes=np.array([(o.nv, o.nt) for o in s.outs], np.int32))
    if form == "stitch":
        nv, nt = C.c_int32(), C.c_int32()
        mesher.check(mesher.lib().lvn_generate_seam_mesh(
            s.ctx._h, abi.vptr(s.min), s.size, C.cast(s.srcs, C.c_void_p), len(s.nodes), abi.vptr(s.colour),
            s.v.data_ptr(), len(s.v), C.byref(nv), s.t.data_ptr(), len(s.t), C.byref(nt)), "seam")
        return dict(vertices=s.v, triangles=s.t, filled=np.array([nv.value, nt.value], np.int32))
    # serve: a burst, its meshes, then a burst elsewhere
    m, said = _Mesh(s), []
    for mins, sizes in s.lists:
        tickets = s.server.submit_meshes(mins, sizes)
        s.server.drain()
        done = np.sort(s.server.poll(2 * len(tickets)), order="ticket")
        said.append(np.stack([done[c] for c in ("status", "nv", "nt", "ns")], axis=1))
        for ticket, r in zip(tickets, done):
            if r["ns"] or r["nv"]:
                m.call(mesher.lib().lvn_server_get_mesh, s.server._h, int(ticket))
    return dict(_meshes(s, m.at), served=said)


# ---------------------------------------------------------------- what a pass cannot do without

SNOISE2, SNOISE3 = 49, 87  # operations of one noise evaluation (fused multiply-add = 2)


def work(case):
    """Every field column and (with caves) sample evaluated once, 23 field evaluations per
    crossing edge as the method defines them; every mesh written once."""
    _enter(case)
    d = workloads.heightfield_desc() if case["field"] == "height" else workloads.terrain_desc()
    height = 14 * SNOISE2 + 117 if case["field"] == "leven" else 3 + (SNOISE2 + 5) * d.height_octaves
    cave = 5 + (SNOISE3 + 6) * d.cave_octaves if case["field"] == "caves" else 0
    seed, form = 1, case["form"]
    if form == "stitch":
        s = prepare(case, seed)
        out = run(s)
        offered = sum(len(l["nodes"]) for l in s.nodes)
        return dict(bytes=48 * (offered + int(out["filled"][0])) + 12 * int(out["filled"][1]), flops=0)
    if form in ("chunk", "scratch", "edit"):
        size = _size(case)
        mins, sizes = [_column(case, seed, size)], [size]
    else:
        mins, sizes = _place(case if form != "serve" else dict(case, near=2 * case["near"]), seed)
    k = np.zeros((0, 6), np.int64)
    for i in range(0, len(sizes), 256):
        k = np.concatenate([k, _count(case, mins[i:i + 256], sizes[i:i + 256])])
    e, v, t, q = (int(x) for x in k[:, :4].sum(axis=0))
    f = case["voxels"] + 2
    mesh = 48 * v + 12 * t + 48 * q
    flops = len(sizes) * (f * f * height + f ** 3 * cave) + 23 * e * (height + cave)
    if form == "edit":  # the field is kept: the brushes' edges only, and two meshes
        return dict(bytes=2 * (f ** 3 + mesh), flops=2 * 1000 * v)
    if form == "simplify":
        mesh *= 3
    return dict(bytes=mesh, flops=flops)


# ---------------------------------------------------------------- 64-bit values

def _noise2(table, px, py):
    """Simplex noise over the permutation table (texel value's low four bits pick the gradient)."""
    g3 = np.array([[0, 1], [0, 1], [0, -1], [0, -1], [1, 0], [1, 0], [-1, 0], [-1, 0], [1, 1], [1, -1], [-1, 1],
                   [-1, -1], [1, 0], [-1, 0], [0, -1], [0, 1]])
    grad = (g3 * 64 + 64) / 255.0 * 4.0 - 1.0
    f2, g2 = 0.366025403784, 0.211324865405
    s = (px + py) * f2
    ix, iy = np.floor(px + s), np.floor(py + s)
    t = (ix + iy) * g2
    fx, fy = px - (ix - t), py - (iy - t)
    ox = (fx > fy).astype(int)
    total = 0.0
    for dx, dy, x, y in ((0, 0, fx, fy), (ox, 1 - ox, fx - ox + g2, fy - (1 - ox) + g2),
                         (1, 1, fx - 1 + 2 * g2, fy - 1 + 2 * g2)):
        g = grad[table[(iy.astype(int) + dy) & 255, (ix.astype(int) + dx) & 255] & 15]
        total = total + np.maximum(0.5 - x * x - y * y, 0.0) ** 4 * (g[..., 0] * x + g[..., 1] * y)
    return 70.0 * total


def exact(case, seed):
    """Vertices of one heightfield chunk without brushes, in 64 bits: density, the 17-sample
    crossing, central-difference normals and the truncated least-squares vertex.  The other
    fields have no such value: whether a sample lies inside is the sign of a 32-bit sum of
    900 voxels or of aliased octaves, so 64 bits give other voxels, in other places.  The
    permutation table is an input, read where a program reads it."""
    if case["form"] not in ("chunk", "scratch") or case["field"] != "height" or case["brushes"]:
        return None
    if case.get("flags", 0):
        return None
    _enter(case)
    size, n = _size(case), case["voxels"]
    lo = np.array(_column(case, seed, size))
    table, off, scale = mesher.perm_table().reshape(256, 256).astype(int), lo // 4, size // (4 * n)

    def height(x, z):
        total, f, amp = 0.0, 1.0 / 128.0, 24.0
        for _ in range(6):
            total, f, amp = total + amp * _noise2(table, x * f, z * f), f * 2.0, amp * 0.5
        return total

    w = [off[a] + scale * np.arange(n + 2.0) for a in range(3)]
    top = height(w[0][None, :], w[2][:, None])                     # [z, x]
    solid = (w[1][None, :, None] - top[:, None, :]) < 0.0           # [z, y, x]
    ident, point, h = {}, [], 0.001
    o = solid[:-1, :-1, :-1]
    for z, y, x in np.argwhere((o != solid[:-1, :-1, 1:]) | (o != solid[:-1, 1:, :-1]) | (o != solid[1:, :-1, :-1])):
        for axis, (dz, dy, dx) in enumerate(((0, 0, 1), (0, 1, 0), (1, 0, 0))):
            if solid[z, y, x] != solid[z + dz, y + dy, x + dx]:
                ident[x, y, z, axis] = len(point)
                point.append((x, y, z, axis))
    if not point:
        return None
    p = np.array(point)
    step = np.eye(3)[p[:, 3]]
    base = off + scale * p[:, :3]
    t = np.arange(17) / 16.0
    at = base[:, None, :] + scale * t[None, :, None] * step[:, None, :]
    k = np.argmin(np.abs(at[..., 1] - height(at[..., 0], at[..., 2])), axis=1)
    q = base + scale * (t[k, None] * step)
    grad = np.stack([height(q[:, 0] - h, q[:, 2]) - height(q[:, 0] + h, q[:, 2]), np.full(len(q), 2 * h),
                     height(q[:, 0], q[:, 2] - h) - height(q[:, 0], q[:, 2] + h)], axis=1)
    normal = grad / np.linalg.norm(grad, axis=1, keepdims=True)
    local = scale * (p[:, :3] + t[k, None] * step)
    corners = np.stack([solid[dz:n + dz, dy:n + dy, dx:n + dx] for dz in (0, 1) for dy in (0, 1) for dx in (0, 1)])
    active = np.argwhere(corners.any(axis=0) & ~corners.all(axis=0))
    rgb = {256: (0.3, 0.1, 0.0), 512: (0.0, 0.0, 0.5), 1024: (0.0, 0.5, 0.5), 2048: (0.5, 0.0, 0.5),
           4096: (0.0, 0.5, 0.0)}
    colour = next((c for s, c in rgb.items() if size // 256 == s // 256), (0.5, 0.0, 0.0))
    out = np.zeros((_rows(case, 1)[0], 12))
    for i, (z, y, x) in enumerate(active):
        own = [ident.get(key, -1) for b in (0, 1) for a in (0, 1) for key in
               ((x, y + a, z + b, 0), (x + a, y, z + b, 1), (x + a, y + b, z, 2))]
        own = [e for e in own if e >= 0]
        m, nn = local[own].mean(axis=0), normal[own]
        val, vec = np.linalg.eigh(nn.T @ nn)
        keep = (np.abs(val) >= 0.1) & (np.abs(val) <= 10.0)
        inv = np.where(keep, 1.0 / np.where(keep, val, 1.0), 0.0)
        r = nn.T @ ((local[own] - m) * nn).sum(axis=1)
        out[i, :3] = 4.0 * (vec @ (inv * (vec.T @ r)) + m) + lo
        out[i, 3] = 1.0
        out[i, 4:7] = nn.mean(axis=0)
        out[i, 8:11] = colour
    return dict(vertices=out, triangles=None, seam_voxels=None, seam_points=None, filled=None)
