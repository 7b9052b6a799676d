"""The work whose time counts: what a program that uses this library has it do, at the sizes it does it.

listed() names the cases, draw() gives others of the same ranges, prepare() makes what the program
holds before the call (buffers, geometry, accels), run() is one pass through the public entry points,
work() what a pass cannot do without and exact() the same outputs from 64-bit torch.

Families, by the entry point a pass goes through:
  scan    gprtBufferExclusiveSum / Partition / Select over 32-bit items
  sort    gprtBufferSort, gprtBufferSortPayload (64-bit) and the width-explicit sorts; the pass copies
          the unsorted keys in first, as a program that sorts new keys every time writes them
  scene   gprtAccelBuild, then gprtAccelTraceClosestHit: a small interactive scene, triangles or boxes
  build   gprtAccelBuild of one triangle mesh, a soup or an indexed surface
  update  gprtAccelUpdate (refit) of a mesh whose vertices have moved since it was built
  trace   gprtAccelTraceClosestHit of primary and bounce rays through a built scene
  batch   gprtAccelBuildBatch of many uneven meshes
  frame   an animated frame: every mesh moved and rebuilt, the instance accel rebuilt over them,
          primary rays traced, bounce rays made from their hits and traced
  train   gprtProposalTrainLabels from a given checkpoint: one epoch, and the weights read back
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gprt_amd import api, scenes

DEV = "cuda"
FAR = 100.0  # the rays' far end: scenes lie within a few units of the unit cube


# ------------------------------------------------------------------------------------------------
# Cases
# ------------------------------------------------------------------------------------------------
def listed():
    return [
        # A thousand per-object counts to offsets: the smallest call, all latency.
        {"name": "sum_small", "family": "scan", "op": "sum", "n": 1_000},
        # The 10^8-element buffers of the buffer tests, with a ragged end.
        {"name": "sum_large", "family": "scan", "op": "sum", "n": 99_999_999},
        # Stream compaction of one large wavefront of rays or particles by sign.
        {"name": "partition_mid", "family": "scan", "op": "partition", "n": 10_000_001},
        # A few thousand 64-bit keys with payload (GPRT's own sort entry point): draw lists, small grids.
        {"name": "sort_small", "family": "sort", "n": 3_000, "key": 64, "value": 64, "bits": 64},
        # The sort microbenchmark: 2^26 32-bit keys with 32-bit payload.
        {"name": "sort_large", "family": "sort", "n": 1 << 26, "key": 32, "value": 32, "bits": 32},
        # The smallest scene of the benchmark configurations: 16,384 triangles, 256 x 256 rays.
        {"name": "scene_small", "family": "scene", "kind": "triangles", "n": 16_384, "rays": 65_536},
        # The large scene's build.
        {"name": "build_large", "family": "build", "mesh": "soup", "n": 4_194_304},
        # A deforming character or cloth: an indexed surface, refit every frame.
        {"name": "update_mid", "family": "update", "mesh": "indexed", "n": 999_999},
        # The large scene's rays: 2048 x 2048 primary and as many bounce rays.
        {"name": "trace_large", "family": "trace", "n": 4_194_304, "side": 2_048},
        # A level's worth of meshes, log-uniform in size as in the batched benchmark.
        {"name": "batch_mid", "family": "batch", "meshes": 1_000, "low": 64, "high": 65_536},
        # The dynamic scene: 64 meshes of 65,536 triangles, 1024 x 1024 primary and bounce rays.
        {"name": "frame_large", "family": "frame", "meshes": 64, "per": 65_536, "side": 1_024, "placed": False},
        # Fine-tuning the proposal on a frame's rays with the bindings' default batch.
        {"name": "train_mid", "family": "train", "rays": 131_072, "batch": 8_192},
    ]


def _size(rng, low, high):
    """Log-uniform in [low, high], rarely round."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    family = rng.choice(["scan", "scan", "sort", "sort", "scene", "build", "update", "trace", "batch", "frame", "train"])
    if family == "scan":
        return {"family": family, "op": rng.choice(["sum", "partition", "select"]), "n": _size(rng, 1_000, 99_999_999)}
    if family == "sort":
        key, value = rng.choice([(64, 64), (64, 0), (32, 32), (32, 0), (64, 32)])
        bits = rng.choice([key, key, 30 if key == 32 else 48])  # cell and Morton keys leave the high bits 0
        return {"family": family, "n": _size(rng, 3_000, (1 << 26) * 64 // (key + value) // (key // 32)), "key": key,
                "value": value, "bits": bits}
    if family == "scene":
        return {"family": family, "kind": rng.choice(["triangles", "boxes"]), "n": _size(rng, 500, 1_000_000),
                "rays": _size(rng, 1_000, 1_000_000)}
    if family in ("build", "update"):
        return {"family": family, "mesh": rng.choice(["soup", "indexed"]), "n": _size(rng, 20_000, 4_194_304)}
    if family == "trace":
        return {"family": family, "n": _size(rng, 50_000, 4_194_304), "side": _size(rng, 128, 2_048)}
    if family == "batch":
        return {"family": family, "meshes": _size(rng, 16, 1_000), "low": 64, "high": _size(rng, 4_096, 65_536)}
    if family == "frame":
        return {"family": family, "meshes": _size(rng, 4, 64), "per": _size(rng, 2_048, 65_536),
                "side": _size(rng, 128, 1_024), "placed": rng.random() < 0.5}
    return {"family": family, "rays": _size(rng, 8_192, 131_072), "batch": rng.choice([4_096, 8_192])}


# ------------------------------------------------------------------------------------------------
# Buffers and accels that release themselves, and tensors over their memory
# ------------------------------------------------------------------------------------------------
_context = None


def context():
    """The program's one context."""
    global _context
    if _context is None:
        _context = api.Context(0)
    return _context


class _Owned:
    """Keeps a library object, and what it reads, until nothing refers to it any more."""

    def __init__(self, thing, *reads):
        self.thing, self.reads = thing, reads

    def __del__(self):
        self.thing.destroy()


class _Memory:
    def __init__(self, owner, address, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (int(address), False),
                                         "version": 2}


_KINDS = {torch.int32: "<i4", torch.int64: "<i8", torch.float32: "<f4"}


def _tensor(owner, address, shape, dtype):
    return torch.as_tensor(_Memory(owner, address, shape, _KINDS[dtype]), device=DEV)


def buffer(shape, dtype, data=None):
    """(a device buffer, the tensor over it) of one shape and type, filled with `data`."""
    ctx = context()
    shape = (shape,) if isinstance(shape, int) else tuple(shape)
    own = _Owned(ctx.device_buffer(nbytes=math.prod(shape) * torch.empty(0, dtype=dtype).element_size()))
    view = _tensor(own, ctx.lib.gprtBufferGetDevicePointer(own.thing.h, 0), shape, dtype)
    if data is not None:
        view.copy_(data)
    return own, view


def _tree(own, accel, inner, prims):
    """The inner nodes and leaf records of a built accel, through the descriptor its address names
    (AccelDescriptor of gprt_hip_device.h: nodes, records, ...)."""
    at = context().lib.gprtAccelGetDeviceAddress(accel.h, 0)
    nodes, records = _tensor(own, at, (8,), torch.int64)[:2].tolist()
    return {"nodes": _tensor(own, nodes, (inner, 16), torch.int32), "records": _tensor(own, records, (prims, 12), torch.int32)}


def _hits_of(view):
    whole = view.view(torch.int32)
    return {"t": view[:, 0], "prim": whole[:, 1], "uv": view[:, 2:]}


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


# ------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------
def _keys(case, seed):
    g = _generator(seed)
    n, width = case["n"], case["key"]
    high = torch.randint(0, 1 << 32, (n,), generator=g, device=DEV, dtype=torch.int64)
    if width == 32:
        keys = (high & ((1 << case["bits"]) - 1)).to(torch.int32)
    else:
        low = torch.randint(0, 1 << 32, (n,), generator=g, device=DEV, dtype=torch.int64)
        keys = ((high << 32) | low) & (((1 << case["bits"]) - 1) if case["bits"] < 64 else -1)
    values = None
    if case["value"]:
        values = torch.arange(n, device=DEV, dtype=torch.int64).to(torch.int32 if case["value"] == 32 else torch.int64)
    return keys, values


def _items(case, seed):
    g = _generator(seed)
    if case["op"] == "sum":  # counts per object or cell
        return torch.randint(0, 16, (case["n"],), generator=g, device=DEV, dtype=torch.int32)
    return torch.randint(-(1 << 31), 1 << 31, (case["n"],), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)


def _scene_prims(case, seed):
    """Triangles [n, 3, 3] or boxes [n, 2, 3] spread over the unit cube, float32."""
    g = _generator(seed)
    n = case["n"]
    reach = 0.01 * max(1.0, (16_384 / n) ** (1 / 3))
    centre = _uniform(g, n, 1, 3)
    if case["kind"] == "boxes":
        half = _uniform(g, n, 1, 3) * reach
        return torch.cat([centre - half, centre + half], 1).float()
    return (centre + (_uniform(g, n, 3, 3) * 2 - 1) * reach).float()


def _scene_rays(case, seed):
    """Rays [m, 8] {origin, tmin, direction, tmax}: a camera's, and from a quarter on random ones."""
    g = _generator(seed + 77)
    m = case["rays"]
    side = math.isqrt(m - 1) + 1
    k = torch.arange(m, device=DEV, dtype=torch.float64)
    half = math.tan(math.radians(30.0))
    rays = torch.zeros(m, 8, device=DEV, dtype=torch.float64)
    rays[:, 0], rays[:, 1], rays[:, 2] = 0.5, 0.5, -1.0
    rays[:, 4] = ((k % side + 0.5) / side * 2 - 1) * half
    rays[:, 5] = ((torch.div(k, side, rounding_mode="floor") + 0.5) / side * 2 - 1) * half
    rays[:, 6] = 1.0
    loose = m - m // 4
    rays[loose:, :3] = _uniform(g, m - loose, 3) * 2 - 0.5
    rays[loose:, 4:7] = torch.randn(m - loose, 3, generator=g, device=DEV, dtype=torch.float64)
    rays[:, 4:7] /= rays[:, 4:7].norm(dim=1, keepdim=True)
    rays[:, 7] = FAR
    return rays.float()


def _pinhole(side):
    rays = torch.from_numpy(scenes.pinhole_rays(side, side).view(np.float32).reshape(-1, 8).copy())
    rays[:, 7] = FAR
    return rays


def _mesh(case, seed):
    """(vertex buffer, its tensor, index buffer, vertices, triangles): blobs of loose triangles, or a bumpy
    surface on a grid whose triangles share their vertices."""
    ctx, n = context(), case["n"]
    if case["mesh"] == "soup":
        vb, ib = api.synth_blob_meshes(ctx, np.array([n]), seed)
        verts, index = _Owned(vb), _Owned(ib)
        view = _tensor(verts, ctx.lib.gprtBufferGetDevicePointer(vb.h, 0), (3 * n, 3), torch.float32)
        return verts, view, index, 3 * n, n
    g = _generator(seed)
    w = max(1, math.isqrt(n // 2))
    h = -(-n // (2 * w))
    x, y = torch.meshgrid(torch.arange(w + 1, device=DEV), torch.arange(h + 1, device=DEV), indexing="xy")
    x, y = x.reshape(-1).double() / w, y.reshape(-1).double() / h
    wave = _uniform(g, 4, 4)
    z = sum(0.1 * a * torch.sin(2 * math.pi * (b * 6 * x + c * 6 * y + d)) for a, b, c, d in wave)
    verts, view = buffer((x.numel(), 3), torch.float32, torch.stack([x, y, z + 0.5], 1))
    cell = torch.arange(w * h, device=DEV, dtype=torch.int64)
    a = torch.div(cell, w, rounding_mode="floor") * (w + 1) + cell % w
    tri = torch.stack([a, a + 1, a + w + 1, a + 1, a + w + 2, a + w + 1], 1).reshape(-1, 3)[:n]
    index, _ = buffer((n, 3), torch.int32, tri.to(torch.int32))
    return verts, view, index, x.numel(), n


def _placements(count, seed):
    """Rotated, scaled and shifted 3 x 4 transforms."""
    rng = np.random.default_rng(seed)
    out = np.zeros((count, 3, 4), dtype=np.float32)
    for k in range(count):
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        a = q * rng.uniform(0.5, 1.5)
        out[k, :, :3] = a
        out[k, :, 3] = 0.5 - a @ np.full(3, 0.5) + rng.uniform(-0.2, 0.2, 3)
    return out


INPUTS, HIDDEN, CLASSES, BANDS = 102, 128, 4_096, 8


def _checkpoint(seed):
    """He-uniform weights in the library's flat layout W1t b1 W2t b2 W3t b3 W4t b4, float32 on the host."""
    g = torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)
    flat = []
    for rows, fan in ((HIDDEN, INPUTS), (HIDDEN, HIDDEN), (HIDDEN, HIDDEN), (CLASSES, HIDDEN)):
        w = torch.zeros(rows, HIDDEN)
        w[:, :fan] = (torch.rand(rows, fan, generator=g) * 2 - 1) * math.sqrt(6.0 / fan)
        flat += [w.reshape(-1), torch.zeros(rows)]
    return torch.cat(flat).numpy()


def _training_rays(case, seed):
    """(rays [m, 8], labels [m]): rays from in front of the scene and the cell (of 64 x 64) of its middle
    plane that they cross, -1 where they pass beside it."""
    g = _generator(seed)
    m = case["rays"]
    rays = torch.zeros(m, 8, device=DEV, dtype=torch.float64)
    rays[:, :3] = torch.tensor([0.5, 0.5, -1.0], device=DEV, dtype=torch.float64) + (_uniform(g, m, 3) - 0.5) * 0.2
    to = torch.cat([_uniform(g, m, 2) * 1.2 - 0.1, torch.full((m, 1), 0.5, device=DEV, dtype=torch.float64)], 1)
    rays[:, 4:7] = to - rays[:, :3]
    rays[:, 4:7] /= rays[:, 4:7].norm(dim=1, keepdim=True)
    rays[:, 7] = FAR
    cell = torch.floor(to[:, :2] * 64).long()
    inside = ((cell >= 0) & (cell < 64)).all(1)
    return rays.float(), torch.where(inside, cell[:, 1] * 64 + cell[:, 0], -1).to(torch.int32)


# ------------------------------------------------------------------------------------------------
# prepare / run, family by family
# ------------------------------------------------------------------------------------------------
def _prepare_scan(case, seed):
    items, _ = buffer(case["n"], torch.int32, _items(case, seed))
    out, view = buffer(case["n"], torch.int32)
    view.zero_()
    return {"in": items, "out": out, "view": view}


def _run_scan(s):
    lib, c, case = context().lib, context().h, s["case"]
    i, o = s["in"].thing.h, s["out"].thing.h
    if case["op"] == "sum":
        return {"total": int(lib.gprtBufferExclusiveSum(c, i, o, None)), "out": s["view"]}
    if case["op"] == "partition":
        return {"total": int(lib.gprtBufferPartition(c, i, True, o, None)), "out": s["view"]}
    # past the selected items the output keeps what prepare() put there
    return {"total": int(lib.gprtBufferSelect(c, i, True, o, None)), "out": s["view"]}


def _prepare_sort(case, seed):
    keys, values = _keys(case, seed)
    s = {"src": buffer(case["n"], keys.dtype, keys)[0]}
    s["keys"], s["view"] = buffer(case["n"], keys.dtype)
    if values is not None:
        s["vsrc"] = buffer(case["n"], values.dtype, values)[0]
        s["values"], s["vview"] = buffer(case["n"], values.dtype)
    return s


def _run_sort(s):
    lib, c, case = context().lib, context().h, s["case"]
    n, width, value = case["n"], case["key"], case["value"]
    k = s["keys"].thing.h
    lib.gprtBufferCopy(c, s["src"].thing.h, k, 0, 0, width // 8, n, 0, 0)
    out = {"keys": s["view"]}
    if value:
        v = s["values"].thing.h
        lib.gprtBufferCopy(c, s["vsrc"].thing.h, v, 0, 0, value // 8, n, 0, 0)
        out["values"] = s["vview"]
    if not value:
        (lib.gprtBufferSort32 if width == 32 else lib.gprtBufferSort)(c, k, None)
    elif width == value:
        (lib.gprtBufferSortPayload32 if width == 32 else lib.gprtBufferSortPayload)(c, k, v, None)
    else:
        lib.gprtBufferSortKV(c, k, v, n, width, value, None)
    return out


class _Boxes(api.AABBAccel):
    """An AABB accel over boxes that are on the device already."""

    def __init__(self, ctx, boxes, n):
        self.ctx, self.lib, self.nt = ctx, ctx.lib, n
        self.gtype = self.lib.gprtGeomTypeCreate(ctx.h, api.GPRT_AABBS, 0)
        self.geom = self.lib.gprtGeomCreate(ctx.h, self.gtype)
        self.lib.gprtAABBsSetPositions(self.geom, boxes.h, n, 24, 0)
        self.h = self.lib.gprtAABBAccelCreate(ctx.h, self.geom, 0)

    def destroy(self):
        if self.h:
            self.lib.gprtAccelDestroy(self.h)
            self.lib.gprtGeomDestroy(self.geom)
            self.lib.gprtGeomTypeDestroy(self.gtype)
            self.h = None


def _prepare_scene(case, seed):
    ctx, n, m = context(), case["n"], case["rays"]
    prims = _scene_prims(case, seed)
    if case["kind"] == "boxes":
        boxes, _ = buffer((n, 6), torch.float32, prims.reshape(n, 6))
        torch.cuda.synchronize()
        accel = _Owned(_Boxes(ctx, boxes.thing, n), boxes)
    else:
        verts, _ = buffer((3 * n, 3), torch.float32, prims.reshape(3 * n, 3))
        index, _ = buffer(3 * n, torch.int32, torch.arange(3 * n, device=DEV, dtype=torch.int32))
        torch.cuda.synchronize()
        accel = _Owned(api.TriangleAccel(ctx, buffers=(verts.thing, index.thing, 3 * n, n), owns_buffers=False), verts, index)
    accel.thing.build()
    rays, _ = buffer((m, 8), torch.float32, _scene_rays(case, seed))
    hits, view = buffer((m, 4), torch.float32)
    return {"accel": accel, "rays": rays, "hits": hits, "view": view, "tree": _tree(accel, accel.thing, n - 1, n)}


def _run_scene(s):
    s["accel"].thing.build()
    s["accel"].thing.trace(s["rays"].thing, s["hits"].thing, s["case"]["rays"])
    return {**_hits_of(s["view"]), **s["tree"]}


def _prepare_build(case, seed, mode=api.GPRT_BUILD_MODE_FAST_TRACE_NO_UPDATE):
    verts, view, index, nv, n = _mesh(case, seed)
    torch.cuda.synchronize()
    accel = _Owned(api.TriangleAccel(context(), buffers=(verts.thing, index.thing, nv, n), owns_buffers=False), verts, index)
    accel.thing.build(mode)
    return {"accel": accel, "verts": view, "tree": _tree(accel, accel.thing, n - 1, n)}


def _run_build(s):
    s["accel"].thing.build()
    return s["tree"]


def _prepare_update(case, seed):
    s = _prepare_build(case, seed, api.GPRT_BUILD_MODE_FAST_TRACE_AND_UPDATE)
    context().sync()
    g = _generator(seed + 1)
    v = s["verts"]
    v += (torch.rand(v.shape, generator=g, device=DEV) * 2 - 1) * 1e-3
    return s


def _run_update(s):
    s["accel"].thing.update()
    return s["tree"]


def _prepare_trace(case, seed):
    ctx, side = context(), case["side"]
    verts, _, index, nv, n = _mesh({"mesh": "soup", "n": case["n"]}, seed)
    accel = _Owned(api.TriangleAccel(ctx, buffers=(verts.thing, index.thing, nv, n), owns_buffers=False), verts, index)
    accel.thing.build()
    m = side * side
    rays, every = buffer((2 * m, 8), torch.float32)
    hits, view = buffer((2 * m, 4), torch.float32)
    every[:m] = _pinhole(side).to(DEV)
    torch.cuda.synchronize()
    accel.thing.trace(rays.thing, hits.thing, m)
    bounce, made = buffer((m, 8), torch.float32)
    api.bounce_rays(ctx, accel.thing, rays.thing, hits.thing, None, m, bounce.thing, m, seed)
    ctx.sync()
    made[:, 7] = FAR
    every[m:] = made
    torch.cuda.synchronize()
    return {"accel": accel, "rays": rays, "hits": hits, "view": view}


def _run_trace(s):
    s["accel"].thing.trace(s["rays"].thing, s["hits"].thing, 2 * s["case"]["side"] ** 2)
    return _hits_of(s["view"])


def _mesh_sizes(case):
    return scenes.batch_sizes(case["meshes"], 3, case["low"], case["high"])


def _prepare_meshes(ctx, sizes, seed, move):
    vb, ib = api.synth_blob_meshes(ctx, sizes, seed)
    base, index = _Owned(vb), _Owned(ib)
    verts = _Owned(ctx.device_buffer(nbytes=vb.nbytes)) if move else base
    if move:
        ctx.lib.gprtSynthPerturb(ctx.h, vb.h, verts.thing.h, vb.nbytes // 4, seed, 1e-3)
    accels = [_Owned(a, verts, index) for a in api.mesh_accels(ctx, verts.thing, ib, sizes)]
    api.build_batch(ctx, [a.thing for a in accels])
    return {"base": base, "verts": verts, "accels": accels}


def _prepare_batch(case, seed):
    sizes = _mesh_sizes(case)
    s = _prepare_meshes(context(), sizes, seed, False)
    # a batch's accels lie one after the other in one store
    total = int(sizes.sum())
    s["tree"] = _tree(s["accels"], s["accels"][0].thing, total - len(sizes), total)
    return s


def _run_batch(s):
    api.build_batch(context(), [a.thing for a in s["accels"]])
    return s["tree"]


def _prepare_frame(case, seed):
    ctx, m = context(), case["side"] ** 2
    s = _prepare_meshes(ctx, np.full(case["meshes"], case["per"], dtype=np.int64), seed, True)
    places = _placements(case["meshes"], seed) if case["placed"] else None
    s["scene"] = _Owned(api.InstanceAccel(ctx, api.instance_records([a.thing for a in s["accels"]], places)), s["accels"])
    s["scene"].thing.build()
    s["rays"], _ = buffer((m, 8), torch.float32, _pinhole(case["side"]))
    s["bounce"], _ = buffer((m, 8), torch.float32)
    for k in ("primary", "second"):
        s[k], s[k + " hits"] = buffer((m, 4), torch.float32)
        s[k + " inst"], s[k + " inst view"] = buffer(m, torch.int32)
    return s


def _run_frame(s):
    ctx, case, seed, m = context(), s["case"], s["seed"], s["case"]["side"] ** 2
    vb = s["base"].thing
    ctx.lib.gprtSynthPerturb(ctx.h, vb.h, s["verts"].thing.h, vb.nbytes // 4, seed + 1, 1e-3)
    api.build_batch(ctx, [a.thing for a in s["accels"]])
    scene = s["scene"].thing
    scene.build()
    api.trace_detail(ctx, scene, s["rays"].thing, s["primary"].thing, m, s["primary inst"].thing)
    api.bounce_rays(ctx, scene, s["rays"].thing, s["primary"].thing, s["primary inst"].thing, m, s["bounce"].thing, m, seed)
    api.trace_detail(ctx, scene, s["bounce"].thing, s["second"].thing, m, s["second inst"].thing)
    return {k: {**_hits_of(s[k + " hits"]), "inst": s[k + " inst view"]} for k in ("primary", "second")}


def _prepare_train(case, seed):
    rays, labels = _training_rays(case, seed)
    s = {"rays": buffer(rays.shape, torch.float32, rays)[0], "labels": buffer(labels.shape, torch.int32, labels)[0]}
    s["net"] = _Owned(api.Proposal(context(), max_batch=case["batch"], seed=1))
    s["checkpoint"] = _checkpoint(seed)
    return s


RATE = 1e-3


def _run_train(s):
    net = s["net"].thing
    net.set_params(s["checkpoint"])
    loss, accuracy = net.train_labels(s["rays"].thing, s["labels"].thing, s["case"]["rays"], 1, RATE)
    return {"loss": loss, "accuracy": accuracy, "weights": net.get_params()}


_FAMILIES = {"scan": (_prepare_scan, _run_scan), "sort": (_prepare_sort, _run_sort), "scene": (_prepare_scene, _run_scene),
             "build": (_prepare_build, _run_build), "update": (_prepare_update, _run_update),
             "trace": (_prepare_trace, _run_trace), "batch": (_prepare_batch, _run_batch),
             "frame": (_prepare_frame, _run_frame), "train": (_prepare_train, _run_train)}


def prepare(case, seed):
    state = _FAMILIES[case["family"]][0](case, int(seed))
    state["case"], state["seed"] = case, int(seed)
    context().sync()
    torch.cuda.synchronize()
    return state


def run(state):
    return _FAMILIES[state["case"]["family"]][1](state)


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------------
NODE, RECORD, RAY, HIT = 64, 48, 32, 16


def work(case):
    f = case["family"]
    if f == "scan":
        n = case["n"]
        return {"bytes": 4 * n + (2 if case["op"] == "select" else 4) * n, "flops": 0}
    if f == "sort":
        return {"bytes": 2 * case["n"] * (case["key"] + case["value"]) // 8, "flops": 0}
    if f == "train":
        # forward, and the gradients of weights and inputs, of the rays that are labelled (1 / 1.2^2 of them)
        weights = 3 * HIDDEN * HIDDEN + HIDDEN * CLASSES
        return {"bytes": case["rays"] * (RAY + 4) + 8 * weights, "flops": 6 * weights * case["rays"] / 1.44}
    if f == "frame":
        n, m = case["meshes"] * case["per"], case["side"] ** 2
        build = n * (36 + 36 + 12 + NODE + RECORD)  # moved, read, and the meshes' trees written
        top = n * (NODE + RECORD)  # the instance accel over them
        return {"bytes": build + top + 2 * m * (RAY + HIT + 4) + n * (NODE + RECORD), "flops": 0}
    tree = NODE + RECORD
    if f == "batch":
        return {"bytes": int(_mesh_sizes(case).sum()) * (48 + tree), "flops": 0}
    n = case["n"]
    if f == "trace":
        return {"bytes": n * tree + 2 * case["side"] ** 2 * (RAY + HIT), "flops": 0}
    if f == "scene":
        prim = 24 if case["kind"] == "boxes" else 48
        return {"bytes": n * (prim + tree) + case["rays"] * (RAY + HIT) + n * tree, "flops": 0}
    vertices = 36 if case["mesh"] == "soup" else 6  # an indexed surface has half a vertex to a triangle
    return {"bytes": n * (vertices + 12 + tree), "flops": 0}


# ------------------------------------------------------------------------------------------------
# The same outputs in 64 bits
# ------------------------------------------------------------------------------------------------
def _exact_triangles(tri, rays):
    """(t, u, v) of the closest of the triangles [n, 3, 3] for each ray, t = FAR and 0, 0 where none is met."""
    o, d, near, far = rays[:, None, :3], rays[:, None, 4:7], rays[:, 3:4], rays[:, 7:8]
    a, e1, e2 = tri[None, :, 0], tri[None, :, 1] - tri[None, :, 0], tri[None, :, 2] - tri[None, :, 0]
    p = torch.linalg.cross(d.expand(-1, len(tri), -1), e2.expand(len(rays), -1, -1))
    det = (e1 * p).sum(-1)
    s = o - a
    u = (s * p).sum(-1) / det
    q = torch.linalg.cross(s, e1.expand(len(rays), -1, -1))
    v = (d * q).sum(-1) / det
    t = (e2 * q).sum(-1) / det
    met = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > near) & (t < far)
    best, k = torch.where(met, t, math.inf).min(1)
    hit = best < math.inf
    # the library's u and v weigh the second and third vertex
    u, v = u.gather(1, k[:, None])[:, 0], v.gather(1, k[:, None])[:, 0]
    zero = torch.zeros_like(u)
    return torch.where(hit, best, far[:, 0]), torch.where(hit, u, zero), torch.where(hit, v, zero)


def _exact_boxes(box, rays):
    o, d, near, far = rays[:, None, :3], rays[:, None, 4:7], rays[:, 3:4], rays[:, 7:8]
    t0, t1 = (box[None, :, 0] - o) / d, (box[None, :, 1] - o) / d
    lo, hi = torch.minimum(t0, t1).amax(-1), torch.maximum(t0, t1).amin(-1)
    t = torch.where(lo > near, lo, hi)
    best = torch.where((lo <= hi) & (t > near) & (t < far), t, math.inf).amin(1)
    best = torch.where(best < math.inf, best, far[:, 0])
    return best, torch.zeros_like(best), torch.zeros_like(best)


def _exact_scene(case, seed):
    if case["n"] * case["rays"] > 1 << 31:
        return None
    prims, rays = _scene_prims(case, seed).double(), _scene_rays(case, seed).double()
    step = max(1, (1 << 22) // case["n"])
    one = _exact_boxes if case["kind"] == "boxes" else _exact_triangles
    t, u, v = (torch.cat(x) for x in zip(*(one(prims, rays[k:k + step]) for k in range(0, len(rays), step))))
    return {"t": t, "prim": None, "uv": torch.stack([u, v], 1), "nodes": None, "records": None}


def _exact_train(case, seed):
    rays, labels = _training_rays(case, seed)
    rays, labels = rays[labels >= 0].double(), labels[labels >= 0].long()
    x = rays[:, [0, 1, 2, 4, 5, 6]]
    wave = x[:, :, None] * (math.pi * 2.0 ** torch.arange(BANDS, device=DEV, dtype=torch.float64))
    x = torch.cat([x, torch.stack([wave.sin(), wave.cos()], 3).reshape(len(x), -1)], 1)
    x = torch.nn.functional.pad(x, (0, HIDDEN - INPUTS))
    flat = torch.from_numpy(_checkpoint(seed)).to(DEV).double()
    m, v = torch.zeros_like(flat), torch.zeros_like(flat)
    b1, b2, eps = 0.9, 0.999, 1e-8
    loss, steps = 0.0, 0
    for k in range(0, len(x), case["batch"]):
        flat = flat.detach().requires_grad_()
        h, at = x[k:k + case["batch"]], 0
        for rows in (HIDDEN, HIDDEN, HIDDEN, CLASSES):
            w, b = flat[at:at + rows * HIDDEN].view(rows, HIDDEN), flat[at + rows * HIDDEN:at + rows * HIDDEN + rows]
            h, at = h @ w.T + b, at + rows * HIDDEN + rows
            h = h.relu() if rows == HIDDEN else h
        one = torch.nn.functional.cross_entropy(h, labels[k:k + case["batch"]])
        grad, = torch.autograd.grad(one, flat)
        loss, steps = loss + float(one), steps + 1
        with torch.no_grad():
            m, v = b1 * m + (1 - b1) * grad, b2 * v + (1 - b2) * grad * grad
            flat = flat - RATE * (m / (1 - b1 ** steps)) / ((v / (1 - b2 ** steps)).sqrt() + eps)
    return {"loss": loss / max(1, steps), "accuracy": None, "weights": flat.detach()}


def exact(case, seed):
    if case["family"] == "scene":
        return _exact_scene(case, int(seed))
    if case["family"] == "train":
        return _exact_train(case, int(seed))
    return None
