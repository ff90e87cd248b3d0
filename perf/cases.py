"""The work a user of the rasterizer has it do, as cases that can be timed.

Every case goes through the package's public entry points (the Renderer,
BinModel and render_batch classes over the C ABI of include/rast.h):

  frame    one camera's frame: render, then the device pointers of vis,
           depth and RGBA8 (a zero-copy consumer); cameras follow a path
  present  the same, but RGBA8 copied to host memory (a window or a file)
  views    several views of one scene in one launch (main view + cube map, or
           an object from many sides)
  train    the learned capacity model's training over recorded frames
  forward  the model's predictions for host data in a serving loop

A case is a dict of plain values; prepare() makes its inputs from the seed
(terrain heights, placements, cameras, texture offsets, sample values), run()
is one pass.  Scene sizes are those of the package's own workloads and tests.
"""
from __future__ import annotations

import ctypes as C
import functools
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "custom-gpgpu-rasterizer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import autotune  # noqa: E402
import rast as R  # noqa: E402
import scenes as S  # noqa: E402

POLICIES = {"exact": R.BIN_EXACT, "learned": R.BIN_LEARNED, "prevframe": R.BIN_PREVFRAME}
PATH = 16         # cameras of a path, visited in turn
MODEL_FRAMES = 8  # frames a capacity model is trained on before a learned case


# ------------------------------------------------------------------- cases

def _frame(name, scene, size, width, height, **kw):
    c = {"name": name, "kind": "frame", "scene": scene, "size": size, "width": width, "height": height,
         "policy": "exact", "sample": 0, "visual": 0, "cull": 0, "maps": 4, "tex": 2048, "graph": False,
         "shade": True}
    c.update(kw)
    return c


def listed():
    return [
        # one small object in a small window: launches and latency
        _frame("frame_sphere_480p", "sphere", 32, 640, 480, maps=1, tex=256),
        # a thumbnail-sized frame of strips and vertex colours beside textured
        # lists, both faces, filtered, replayed from a graph
        _frame("frame_mixed_431p", "mixed", 40, 777, 431, sample=1, cull=2, tex=512, graph=True),
        # many instanced dense meshes in full HD: sub-pixel triangles
        _frame("frame_icospheres_1080p", "icospheres", 16, 1920, 1080),
        # the large terrain in 4K with learned single-pass binning, moving camera
        _frame("frame_terrain_4k", "terrain", 1024, 3840, 2160, policy="learned"),
        # an odd window size, filtered sampling, previous-frame binning
        _frame("frame_terrain_1439p_linear", "terrain", 700, 2561, 1439, policy="prevframe", sample=1, tex=1024),
        # an 8K still
        _frame("frame_terrain_8k", "terrain", 1024, 7680, 4320),
        # visibility and depth only (a depth pre-pass or shadow map)
        _frame("frame_depth_2k", "icospheres", 8, 2048, 2048, policy="prevframe", shade=False),
        # an interactive window: the frame's colours copied to host memory
        _frame("present_terrain_1080p", "terrain", 512, 1920, 1080, kind="present", tex=1024),
        # a catalogue: thumbnails of one object from 12 sides in one launch
        {"name": "views_turntable_12", "kind": "views", "scene": "object", "size": 6, "views": 12, "width": 256,
         "height": 256, "policy": "exact", "tex": 512},
        # a 4K main view and six cube-map faces of one scene per frame
        {"name": "views_flythrough_7", "kind": "views", "scene": "fly", "size": 1160, "spheres": 64, "width": 3840,
         "height": 2160, "face": 1024, "policy": "learned", "tex": 2048},
        # training the capacity model on a recorded camera path
        {"name": "train_h64", "kind": "train", "hidden": 64, "frames": 12, "width": 3840, "height": 2160, "size": 512,
         "epochs": 2, "batch": 8192},
        # predicting a frame's tiles in a loop that must not allocate
        {"name": "forward_8160", "kind": "forward", "hidden": 64, "samples": 8160},
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    # (views are not drawn: the listed ones are the two uses they have)
    kind = rng.choice(["frame", "frame", "frame", "present", "train", "forward"])
    if kind in ("frame", "present"):
        scene = rng.choice(["sphere", "mixed", "icospheres", "terrain", "terrain"])
        size = {"sphere": lambda: round(log(16, 256)), "mixed": lambda: round(log(16, 160)),
                "icospheres": lambda: round(log(2, 12)), "terrain": lambda: round(log(32, 1024))}[scene]()
        width = round(log(128, 3840))
        height = min(2304, max(64, round(width * rng.uniform(0.4, 1.3))))
        c = _frame("", scene, size, width, height, kind=kind,
                   policy=rng.choice(["exact", "exact", "learned", "prevframe"]), sample=rng.choice([0, 0, 1]),
                   visual=rng.choice([0, 0, 0, 1, 2]), cull=rng.choice([0, 0, 0, 2]),
                   maps=rng.choice([0, 1, 4, 4]), tex=rng.choice([256, 500, 1024]),
                   graph=rng.random() < 0.25, shade=kind == "present" or rng.random() < 0.85)
        del c["name"]
        return c
    if kind == "train":
        return {"kind": "train", "hidden": rng.choice([16, 32, 64]), "frames": rng.randint(2, 12),
                "width": round(log(640, 3840)), "height": round(log(480, 2160)), "size": round(log(100, 512)),
                "epochs": rng.randint(1, 3), "batch": rng.choice([1000, 4096, 8192, 12345])}
    return {"kind": "forward", "hidden": rng.choice([16, 32, 64]), "samples": round(log(1, 65536))}


# ------------------------------------------------------------------ scenes

@functools.lru_cache(maxsize=8)
def _base_maps(size):
    return S.noise_maps(size, S.SEED_BASE + 77)


def _maps(size, seed, count=4):
    """The package's four noise maps shifted by a seeded offset."""
    r = random.Random(seed)
    out = []
    for k in range(4):
        dy, dx = r.randrange(size), r.randrange(size)
        out.append(np.ascontiguousarray(np.roll(_base_maps(size)[k], (dy, dx), (0, 1))) if k < count else None)
    return out if count else None


def _strip(m, n):
    """A terrain of n x n quads as one triangle strip (rows joined by repeated
    indices)."""
    w = n + 1
    rows = []
    for j in range(n):
        top = np.arange(j * w, j * w + w, dtype=np.uint32)
        row = np.stack([top, top + w], 1).ravel()
        rows += [row[:1], row, row[-1:]]
    return S.Mesh(verts=m.verts, indices=np.concatenate(rows), topology=S.TOPO_STRIP)


def _orbit(count, rng, distance):
    yaw, el = rng.uniform(0, 6.28), rng.uniform(-0.7, 0.7)
    return [S.orbit_camera(yaw + 0.05 * k, el, distance) for k in range(count)]


def _scene(case, seed):
    """(scene, camera path) of a frame case."""
    rng = random.Random(seed)
    n, kind, maps = case["size"], case["scene"], case["maps"]
    s32 = rng.randrange(1 << 30)
    if kind == "sphere":
        m = S.uv_sphere(2 * n, n, rng.uniform(0.9, 1.1))
        if maps == 1:
            m.textures = [S.checker(case["tex"], case["tex"], 32), None, None, None]
        else:
            m.textures = _maps(case["tex"], s32, maps)
        return S.Scene([m]), _orbit(PATH, rng, rng.uniform(2.8, 3.2))
    if kind == "terrain":
        path = S.camera_path(s32, 200)[:PATH]
        ter = S.terrain(n, 80.0, 6.0, 6, s32 + 1, 1.0)
        bd = S.backdrop(path[0], case["width"] / case["height"])
        ter.textures = bd.textures = _maps(case["tex"], s32 + 2, maps)
        return S.Scene([ter, bd]), path
    if kind == "icospheres":
        base = S.icosphere(5, 1.0)
        tex = _maps(case["tex"], s32, maps)
        meshes = []
        for j in range(n):
            for i in range(n):
                t = ((i - (n - 1) / 2) * 4.4, ((n - 1) / 2 - j) * 2.5, 0.0)
                e = tuple(rng.uniform(0, 6.2831853) for _ in range(3))
                meshes.append(S.Mesh(verts=base.verts, indices=base.indices,
                                     world=S.world_matrix(t, e, rng.uniform(0.5, 1.5)), textures=tex))
        d = 45.0 * n / 16
        return S.Scene(meshes), [S.Camera(position=(0.02 * k * d / 45, 0.0, d), forward=(0.0, 0.0, 1.0))
                                 for k in range(PATH)]
    # mixed: a strip of vertex colours, and lists with one and four maps (of two sizes)
    path = S.camera_path(s32, 200)[:PATH]
    ground = _strip(S.terrain(n, 80.0, 6.0, 6, s32 + 1, 1.0), n)
    a, b = S.icosphere(4, 1.0), S.uv_sphere(96, 48, 1.0)
    four = _maps(case["tex"], s32 + 2, 4)
    small = _maps(max(16, case["tex"] // 2), s32 + 3, 4)
    a.textures = [four[0], small[1], four[2], small[3]] if maps == 4 else ([four[0], None, None, None] if maps else None)
    b.textures = [four[0], None, None, None] if maps else None
    for m in (a, b):
        m.world = S.world_matrix((rng.uniform(-12, 12), rng.uniform(8, 12), rng.uniform(5, 25)),
                                 tuple(rng.uniform(0, 6.28) for _ in range(3)), rng.uniform(2.0, 5.0))
    return S.Scene([ground, a, b]), path


def _views_scene(case, seed):
    """(scene, per frame the [(camera, width, height)] of its views)."""
    rng = random.Random(seed)
    s32 = rng.randrange(1 << 30)
    maps = _maps(case["tex"], s32, 4)
    if case["scene"] == "object":
        m = S.icosphere(case["size"], 1.0)
        m.world = S.world_matrix((0.0, 0.0, 0.0), tuple(rng.uniform(0, 6.28) for _ in range(3)), rng.uniform(0.9, 1.1))
        m.textures = maps
        n, yaw, el = case["views"], rng.uniform(0, 6.28), rng.uniform(-0.5, 0.5)
        return S.Scene([m]), [[(S.orbit_camera(yaw + 2 * math.pi * (v + k / PATH) / n, el, 3.2), case["width"],
                                case["height"]) for v in range(n)] for k in range(PATH)]
    ter = S.terrain(case["size"], 80.0, 6.0, 6, s32 + 1, 1.0)
    ter.textures = maps
    base = S.icosphere(5, 1.0)
    meshes = [ter]
    for _ in range(case["spheres"]):
        t = (rng.uniform(-34, 34), rng.uniform(7.5, 14), rng.uniform(-34, 34))
        e = tuple(rng.uniform(0, 6.2831853) for _ in range(3))
        meshes.append(S.Mesh(verts=base.verts, indices=base.indices,
                             world=S.world_matrix(t, e, rng.uniform(1.0, 2.5)), textures=maps))
    fly = S.Flythrough(S.Scene(meshes), S.camera_path(s32 + 2, 300)[:PATH], (case["width"], case["height"]),
                       case["face"])
    return fly.scene, [fly.views(f) for f in range(PATH)]


# ------------------------------------------------------------------- state

class Owner:
    """Closes the renderers and models of a state when the state and every
    buffer taken from it are gone."""

    def __init__(self):
        self.models, self.renderers = [], []

    def renderer(self, width, height, tris, of=None):
        r = R.Renderer(width, height) if of is None else of.view(width, height)
        autotune.choose(width, height, tris, _table()).apply(r)
        self.renderers.append(r)
        return r

    def model(self, r, hidden, seed):
        m = R.BinModel(r, hidden=hidden, seed=seed)
        self.models.append(m)
        return m

    def __del__(self):
        for m in self.models:
            m.close()
        for r in reversed(self.renderers):
            r.close()


class Buffer:
    """A device buffer of a frame as the array interface that torch reads."""

    def __init__(self, owner, ptr, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (ptr, False), "version": 2}


@functools.lru_cache(maxsize=1)
def _table():
    return autotune.load_table()


def _buffers(state, r, what=("vis", "depth", "rgba")):
    """The frame's device buffers as tensors (the frame is finished)."""
    p = (C.c_void_p(), C.c_void_p(), C.c_void_p())
    R.check(R.lib().rast_frame_buffers(r.h, *(C.byref(q) for q in p)), "rast_frame_buffers")
    out = {}
    for name, q in zip(("vis", "depth", "rgba"), p):
        if name not in what:
            continue
        key = (q.value, r.width, r.height)
        if key not in state["tensors"]:
            shape, kind = {"vis": ((r.height, r.width), "<i4"), "depth": ((r.height, r.width), "<f4"),
                           "rgba": ((r.height, r.width, 4), "|u1")}[name]
            state["tensors"][key] = torch.as_tensor(Buffer(state["owner"], q.value, shape, kind), device="cuda")
        out[name] = state["tensors"][key]
    return out


def _train_model(owner, r, cams, opts, width, height, tris, seed):
    """A capacity model attached to r, trained briefly on frames of the path."""
    m = owner.model(r, 64, seed)
    m.attach(r, *autotune.queue_depth(width, height, tris, "learned", _table()))
    for k in range(MODEL_FRAMES):
        r.render(cams[k % len(cams)], opts, R.BIN_EXACT, R.FLAG_NO_SHADE)
        if k:
            m.record(r)
    m.train(epochs=8, batch=2048, lr=2e-3, tau=0.95)
    m.clear()


def _prepare_frame(case, seed):
    scene, path = _scene(case, seed)
    owner = Owner()
    W, H, tris = case["width"], case["height"], scene.num_triangles
    r = owner.renderer(W, H, tris)
    r.add_scene(scene)
    opts = S.Opts(cull_mode=case["cull"], sample_state=case["sample"], visualisation=case["visual"])
    if case["policy"] == "learned":
        _train_model(owner, r, path, opts, W, H, tris, 7)
    elif case["policy"] == "prevframe":
        r.set_queue_depth(*autotune.queue_depth(W, H, tris, "prevframe", _table()))
    flags = (R.FLAG_GRAPH if case["graph"] else 0) | (0 if case["shade"] else R.FLAG_NO_SHADE)
    return {"kind": case["kind"], "owner": owner, "r": r, "path": path, "opts": opts,
            "policy": POLICIES[case["policy"]], "flags": flags, "k": 0, "tensors": {},
            "what": ("vis", "depth", "rgba") if case["shade"] else ("vis", "depth")}


def _prepare_views(case, seed):
    scene, frames = _views_scene(case, seed)
    owner, opts, tris = Owner(), S.Opts(), scene.num_triangles
    rs = []
    for _, w, h in frames[0]:
        rs.append(owner.renderer(w, h, tris, of=rs[0] if rs else None))
    rs[0].add_scene(scene)
    if case["policy"] == "learned":  # one model per view, trained briefly
        models = []
        for k, r in enumerate(rs):
            models.append(owner.model(r, 64, 31 + k))
            models[k].attach(r, *autotune.queue_depth(r.width, r.height, tris, "learned", _table()))
        for f in range(4):
            R.render_batch([(r, cam, opts, R.BIN_EXACT, R.FLAG_NO_SHADE) for r, (cam, _, _) in zip(rs, frames[f])])
            if f:
                for m, r in zip(models, rs):
                    m.record(r)
        for m in models:
            m.train(epochs=8, batch=2048, lr=2e-3, tau=0.95)
            m.clear()
    return {"kind": "views", "owner": owner, "rs": rs, "frames": frames, "opts": opts,
            "policy": POLICIES[case["policy"]], "k": 0, "tensors": {}}


def _prepare_train(case, seed):
    frame = _frame("", "terrain", case["size"], case["width"], case["height"], maps=0)
    scene, path = _scene(frame, seed)
    owner = Owner()
    r = owner.renderer(case["width"], case["height"], scene.num_triangles)
    r.add_scene(scene)
    m = owner.model(r, case["hidden"], 1 + seed % 1000003)
    m.attach(r, 1.25, 4)
    for k in range(case["frames"] + 1):
        r.render(path[k % len(path)], S.Opts(), R.BIN_EXACT, R.FLAG_NO_SHADE)
        if k:
            m.record(r)
    return {"kind": "train", "owner": owner, "m": m, "init": m.params(), "epochs": case["epochs"],
            "batch": case["batch"]}


def _forward_inputs(case, seed):
    """Per-tile features: log counts of a tile and its neighbourhoods, min
    depth, tile position; and model weights of trained magnitude."""
    g = np.random.default_rng(seed)
    n, H = case["samples"], case["hidden"]
    x = np.empty((n, 8), np.float32)
    c = np.log1p(np.floor(g.gamma(0.6, 30.0, n)))
    for k in range(5):
        x[:, k] = c if k == 0 else np.maximum(0, c + g.normal(0.2 * k, 0.3, n))
    x[:, 5] = 1.0 - 0.1 * g.random(n) ** 2
    x[:, 6:8] = g.random((n, 2))
    p = [g.uniform(-1, 1, H * 8) * math.sqrt(6 / 8), g.normal(0.01, 0.05, H),
         g.uniform(-1, 1, H * H) * math.sqrt(6 / H), g.normal(0.01, 0.05, H),
         g.uniform(-1, 1, H) * math.sqrt(3 / H), [1.0]]
    return x, np.concatenate(p).astype(np.float32)


def _prepare_forward(case, seed):
    x, p = _forward_inputs(case, seed)
    owner = Owner()
    r = owner.renderer(64, 64, 1000)
    m = owner.model(r, case["hidden"], 1)
    m.set_params(p)
    return {"kind": "forward", "owner": owner, "m": m, "x": x, "pred": np.empty(x.shape[0], np.float32)}


def prepare(case, seed):
    return {"frame": _prepare_frame, "present": _prepare_frame, "views": _prepare_views, "train": _prepare_train,
            "forward": _prepare_forward}[case["kind"]](case, seed)


# --------------------------------------------------------------------- run

def run(state):
    kind = state["kind"]
    if kind in ("frame", "present"):
        k = state["k"]
        state["k"] = (k + 1) % len(state["path"])
        r = state["r"]
        r.render(state["path"][k], state["opts"], state["policy"], state["flags"])
        if kind == "present":
            return {"rgba": r.readback(vis=False, depth=False)[2].view(np.uint8)}
        return _buffers(state, r, state["what"])
    if kind == "views":
        k = state["k"]
        state["k"] = (k + 1) % len(state["frames"])
        R.render_batch([(r, cam, state["opts"], state["policy"], 0)
                        for r, (cam, _, _) in zip(state["rs"], state["frames"][k])])
        return [_buffers(state, r) for r in state["rs"]]
    if kind == "train":
        m = state["m"]
        m.set_params(state["init"])
        loss = m.train(epochs=state["epochs"], batch=state["batch"], lr=2e-3, tau=0.95)
        return {"params": m.params(), "loss": np.float32(loss)}
    m, x, pred = state["m"], state["x"], state["pred"]
    R.check(R.lib().rast_binmodel_forward_noalloc(m.h, x.ctypes.data, x.shape[0], pred.ctypes.data),
            "rast_binmodel_forward_noalloc")
    return {"pred": pred}


# -------------------------------------------------------------------- work

def _geometry(case):
    """(vertices, indices) of a frame case's scene."""
    n = case["size"]
    if case["scene"] == "sphere":
        return (2 * n + 1) * (n + 1), 3 * 2 * n * (2 * n - 1)
    if case["scene"] == "terrain":
        return (n + 1) ** 2 + 24, 6 * n * n + 24
    if case["scene"] == "icospheres":
        return 10242 * n * n, 3 * 20480 * n * n
    return (n + 1) ** 2 + 2562 + 97 * 49, n * (2 * n + 4) + 3 * 5120 + 3 * 96 * 95


def _frame_work(nv, ni, pixels, texels, maps, outputs):
    """Each vertex (56 bytes), index and fetched texel read once, each output
    pixel written once; the arithmetic of the transform (about 120 operations
    a vertex), the triangle setup (100) and the shading (250 a pixel)."""
    b = 56 * nv + 4 * ni + outputs * pixels + 4 * maps * min(texels, pixels)
    return b, 120 * nv + 100 * ni / 3 + 250 * pixels


def work(case):
    kind = case["kind"]
    if kind in ("frame", "present"):
        nv, ni = _geometry(case)
        px = case["width"] * case["height"]
        maps = case["maps"] if case["shade"] and case["visual"] == 0 else 0
        b, f = _frame_work(nv, ni, px, case["tex"] ** 2, maps, 4 if kind == "present" or not case["shade"] else 12)
        if not case["shade"]:
            b += 4 * px
        return {"bytes": b, "flops": f}
    if kind == "views":
        if case["scene"] == "object":
            nv, ni, views = 10 * 4 ** case["size"] + 2, 60 * 4 ** case["size"], case["views"]
            px = views * case["width"] * case["height"]
        else:
            nv = (case["size"] + 1) ** 2 + 10242 * case["spheres"]
            ni = 6 * case["size"] ** 2 + 3 * 20480 * case["spheres"]
            px, views = case["width"] * case["height"] + 6 * case["face"] ** 2, 7
        b, f = _frame_work(nv, ni, px, case["tex"] ** 2, 4, 12)
        return {"bytes": b, "flops": f + (views - 1) * (120 * nv + 100 * ni / 3)}
    H = case["hidden"]
    weights = H * 8 + H * H + H
    if kind == "train":
        tile = autotune.choose(case["width"], case["height"], 2 * case["size"] ** 2 + 8, _table()).tile
        n = case["frames"] * math.ceil(case["width"] / tile) * math.ceil(case["height"] / tile)
        return {"bytes": 36 * n + 8 * weights, "flops": 6 * weights * max(case["batch"], n * case["epochs"])}
    return {"bytes": 36 * case["samples"] + 4 * weights, "flops": 2 * weights * case["samples"]}


# ------------------------------------------------------------------- exact

def _camera64(cam, width, height):
    """View-projection (row, column), camera forward, in 64 bits: look-at
    frame, perspective with the unit [3][3] the frame contract keeps."""
    def unit(v):
        return v / np.linalg.norm(v)

    fwd = unit(np.float64(np.float32(cam.forward)))
    right = unit(np.cross([0.0, 1.0, 0.0], fwd))
    up = unit(np.cross(fwd, right))
    look = np.eye(4)
    look[:3, 0], look[:3, 1], look[:3, 2] = right, up, fwd
    look[:3, 3] = np.float64(np.float32(cam.position))
    n, f = float(np.float32(cam.near_z)), float(np.float32(cam.far_z))
    t = math.tan(math.radians(cam.fov_deg) / 2)
    proj = np.eye(4)
    proj[0, 0], proj[1, 1] = height / (width * t), 1 / t
    proj[2, 2], proj[2, 3], proj[3, 2] = f / (n - f), f * n / (n - f), -1.0
    return proj @ np.linalg.inv(look), fwd


def _triangles64(m, vp, dev):
    """Clip-divided corners of a mesh's triangles: three (n, 3) tensors."""
    world = np.float64(np.asarray(m.world, np.float32)).reshape(4, 4).T
    p = torch.from_numpy(np.float64(m.verts[:, :3])).to(dev)
    M = torch.from_numpy(vp @ world).to(dev)
    c = torch.stack([sum(M[r, k] * p[:, k] for k in range(3)) + M[r, 3] for r in range(4)], 1)
    ndc = c[:, :3] / c[:, 3:]
    ix = torch.from_numpy(m.indices.astype(np.int64)).to(dev)
    if m.topology == S.TOPO_LIST:
        t = ix[:ix.numel() // 3 * 3].view(-1, 3)
    else:
        k = torch.arange(ix.numel() - 2, device=dev)
        odd = k % 2
        t = torch.stack([ix[k], ix[k + 1 + odd], ix[k + 2 - odd]], 1)
    return ndc[t[:, 0]], ndc[t[:, 1]], ndc[t[:, 2]]


def _depth64(scene, cam, width, height, cull):
    """The nearest depth per pixel in 64 bits: every triangle in front of the
    culling rules tested at every pixel of its box."""
    dev = torch.device("cuda")
    vp, fwd = _camera64(cam, width, height)
    out = torch.ones(width * height, dtype=torch.float64, device=dev)
    for m in scene.meshes:
        A, B, D = _triangles64(m, vp, dev)
        ok = torch.isfinite(A).all(1) & torch.isfinite(B).all(1) & torch.isfinite(D).all(1)
        if cull != 2:
            f = torch.cross(B - A, D - A, dim=1)
            cv = sum(float(fwd[k]) * f[:, k] for k in range(3))
            ok &= (cv > 0) if cull == 0 else (cv < 0)
        for k, lo in ((0, -1.0), (1, -1.0), (2, 0.0)):
            lows, highs = torch.stack([A, B, D])[:, :, k], torch.stack([A, B, D])[:, :, k]
            ok &= ~((lows < lo).all(0) | (highs > 1.0).all(0))
        A, B, D = A[ok], B[ok], D[ok]
        x = torch.stack([(q[:, 0] + 1) / 2 * width for q in (A, B, D)], 1)
        y = torch.stack([(1 - q[:, 1]) / 2 * height for q in (A, B, D)], 1)
        z = torch.stack([q[:, 2] for q in (A, B, D)], 1)
        area = ((x[:, 0] - x[:, 1]) * (y[:, 0] - y[:, 2]) - (y[:, 0] - y[:, 1]) * (x[:, 0] - x[:, 2])).abs()
        x0 = x.amin(1).ceil().clamp(0, width).long()
        x1 = x.amax(1).floor().clamp(-1, width - 1).long()
        y0 = y.amin(1).ceil().clamp(0, height).long()
        y1 = y.amax(1).floor().clamp(-1, height - 1).long()
        w, h = (x1 - x0 + 1).clamp_min(0), (y1 - y0 + 1).clamp_min(0)
        items = torch.where(area > 0, w * h, torch.zeros_like(w))
        keep = items > 0
        x, y, z, area, x0, y0, w, items = (q[keep] for q in (x, y, z, area, x0, y0, w, items))
        if not items.numel():
            continue
        # runs of triangles of at most about 2^24 box pixels together
        ends = torch.cumsum(items, 0)
        cuts = torch.unique(torch.searchsorted(ends, torch.arange(0, int(ends[-1]) + 1, 1 << 24, device=dev)))
        edges = sorted(set([0, int(items.numel())] + [int(c) for c in cuts if 0 < c < items.numel()]))
        for lo, hi in zip(edges[:-1], edges[1:]):
            n = items[lo:hi]
            tri = torch.repeat_interleave(torch.arange(lo, hi, device=dev), n)
            q = torch.arange(int(n.sum()), device=dev) - torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
            px, py = x0[tri] + q % w[tri], y0[tri] + q // w[tri]
            zz = torch.zeros_like(px, dtype=torch.float64)
            inside = torch.ones_like(px, dtype=torch.bool)
            for i, j, o in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):  # the edge i -> j weighs corner o
                e = (px - x[tri, i]) * (y[tri, j] - y[tri, i]) - (py - y[tri, i]) * (x[tri, j] - x[tri, i])
                inside &= e >= 0
                zz += e / area[tri] * z[tri, o]
            inside &= (zz >= 0) & (zz <= 1)
            out.scatter_reduce_(0, (py * width + px)[inside], zz[inside], "amin")
    return out.view(height, width).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        scene, path = _scene(case, seed)
        d = _depth64(scene, path[0], case["width"], case["height"], case["cull"])
        return {"vis": None, "depth": d, "rgba": None} if case["shade"] else {"vis": None, "depth": d}
    if kind != "forward":
        # pictures are bytes; training starts from features recorded inside the library
        return None
    x, p = _forward_inputs(case, seed)
    H = case["hidden"]
    x, p = np.float64(x), np.float64(p)
    W1, b1, p = p[:8 * H].reshape(H, 8), p[8 * H:9 * H], p[9 * H:]
    W2, b2, W3, b3 = p[:H * H].reshape(H, H), p[H * H:H * H + H], p[H * H + H:H * H + 2 * H], p[-1]
    h = np.maximum(np.maximum(x @ W1.T + b1, 0) @ W2.T + b2, 0)
    return {"pred": h @ W3 + b3}
