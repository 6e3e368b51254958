"""Performance cases of the render path: what programs have the framework do,
through its public entry points (`axiomr_amd.render`, `.resident`, `.serve`
and the C ABI calls those wrap), from a 512-face object in a 256x256 window to
a 4M-triangle soup at 1080p.

A pass ends as a program's does: with the frames it wanted in host memory,
read into buffers it keeps.  Frames are read with colour and depth (and the
winner keys where the framebuffer has them); images that are the product
themselves (batched views, served requests) with their colour.

Kinds of case:
  scene   one frame of one or several objects, each a drawMesh into the one
          framebuffer, as the application's render loop draws its meshes
  frames  a queue of frames of one large mesh on an orbit, the last one read
          (the repository's benchmark loop)
  soup    one frame of a screen-space triangle soup
  batch   many views in one captured launch
  serve   a burst of requests through the render server

The depth planes have no 64-bit counterpart to be compared with: a pixel on
an edge belongs to another triangle, or to none, in another precision, so
there is no `exact` here.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import axiomr_amd as axr
from axiomr_amd import _native as N
from axiomr_amd import autotune as AT
from axiomr_amd import render as R
from axiomr_amd import resident as RS
from axiomr_amd import scenes as S
from axiomr_amd import serve as SV

SHADERS = ("flat", "phong", "pbr", "gouraud", "phong_point")


def listed():
    return [
        # the smallest call: one 512-face object in a thumbnail window, untuned
        # context, synchronous drawMesh; launches and waits are what counts
        dict(name="small_flat_256", kind="scene", config="default", width=256, height=256, objects=1, shape="uv",
             faces_lo=512, faces_hi=512, shader="flat", bilinear=False, tex=64, groups=1, ids=False, close=False,
             queued=False),
        # the repository's 800x600 UV sphere: Gouraud over a bilinear checker
        dict(name="uv_sphere_800x600", kind="scene", config="default", width=800, height=600, objects=1, shape="uv",
             faces_lo=20000, faces_hi=20000, shader="gouraud", bilinear=True, tex=256, groups=1, ids=False,
             close=False, queued=False),
        # a frame of the application: several meshes with the PBR shader and
        # its five textures, queued draws, an odd window size, untuned context
        dict(name="app_pbr_1241x719", kind="scene", config="default", width=1241, height=719, objects=12, shape="ico",
             faces_lo=2000, faces_hi=60000, shader="pbr", bilinear=True, tex=512, groups=3, ids=False, close=False,
             queued=True),
        # a larger scene under the tuned settings, winner keys kept (picking),
        # nearest texels, synchronous draws
        dict(name="scene_phong_ids_1920x1079", kind="scene", config="plain", width=1920, height=1079, objects=16,
             shape="ico", faces_lo=5000, faces_hi=300000, shader="phong", bilinear=False, tex=1024, groups=2, ids=True,
             close=False, queued=False),
        # a camera among coarse objects: faces across the frustum planes, and
        # triangles that span much of the screen
        dict(name="close_lowpoly_1280x720", kind="scene", config="default", width=1280, height=720, objects=12,
             shape="uv", faces_lo=128, faces_hi=2000, shader="phong_point", bilinear=True, tex=512, groups=1, ids=False,
             close=True, queued=False),
        # the same camera in the tuned settings, with finer meshes
        dict(name="close_mid_1920x1080", kind="scene", config="plain", width=1920, height=1080, objects=8, shape="ico",
             faces_lo=2000, faces_hi=100000, shader="phong_point", bilinear=True, tex=512, groups=1, ids=False,
             close=True, queued=True),
        # the benchmark's 1M-triangle frame at 1080p, queued frames
        dict(name="frames_1M_1080p", kind="frames", config="plain", width=1920, height=1080, n=224, frames=48,
             tex=2048),
        # the overdraw stress, and a soup of ordinary size in an untuned context
        dict(name="soup_4M_1080p", kind="soup", config="soup_4M_1080p", width=1920, height=1080, tris=4_000_000),
        dict(name="soup_150k_1280x720", kind="soup", config="default", width=1280, height=720, tris=150_000),
        # views of shared meshes in one launch: full-size mixed views, and
        # thumbnails of small meshes
        dict(name="batch_40_mixed", kind="batch", config="batch", views=40, meshes=8, f_lo=5000, f_hi=500000, s_lo=256,
             s_hi=1080, tex=1024),
        dict(name="batch_60_thumbnails", kind="batch", config="default", views=60, meshes=12, f_lo=1000, f_hi=20000,
             s_lo=64, s_hi=224, tex=256),
        # a burst of render requests, mixed resolutions
        dict(name="serve_burst_24", kind="serve", config="serve", requests=24, meshes=10, f_lo=10000, f_hi=500000,
             tex=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("scene", "scene", "scene", "frames", "soup", "batch", "serve"))
    config = rng.choice(("default", "plain"))
    if kind == "scene":
        lo = _log(rng, 200, 20000)
        return dict(kind=kind, config=config, width=_log(rng, 128, 1920), height=_log(rng, 96, 1080),
                    objects=rng.randint(1, 16), shape=rng.choice(("uv", "ico")), faces_lo=lo,
                    faces_hi=_log(rng, lo, 200000), shader=rng.choice(SHADERS), bilinear=rng.random() < 0.5,
                    tex=rng.choice((64, 300, 512, 1024)), groups=rng.randint(1, 4), ids=rng.random() < 0.3,
                    close=rng.random() < 0.4, queued=rng.random() < 0.5)
    if kind == "frames":
        return dict(kind=kind, config=config, width=_log(rng, 320, 1920), height=_log(rng, 200, 1080),
                    n=_log(rng, 20, 224), frames=rng.randint(8, 40), tex=rng.choice((256, 1024, 2048)))
    if kind == "soup":
        return dict(kind=kind, config=rng.choice(("default", "plain", "soup_4M_1080p")), width=_log(rng, 320, 1920),
                    height=_log(rng, 200, 1080), tris=_log(rng, 10_000, 4_000_000))
    if kind == "batch":
        lo = _log(rng, 500, 10000)
        s_lo = _log(rng, 64, 300)
        return dict(kind=kind, config=rng.choice(("default", "batch")), views=rng.randint(4, 48),
                    meshes=rng.randint(1, 8), f_lo=lo, f_hi=_log(rng, lo, 400000), s_lo=s_lo,
                    s_hi=_log(rng, s_lo, 900), tex=rng.choice((256, 1024)))
    return dict(kind=kind, config="serve", requests=rng.randint(4, 24), meshes=rng.randint(2, 8), f_lo=5000,
                f_hi=_log(rng, 10000, 500000), tex=rng.choice((256, 1024)))


# ---- what a program keeps ------------------------------------------------------


class _Program:
    """One context with its tunables, and the render server if it serves."""

    def __init__(self, config, served):
        self.ctx = R.Context(0)
        if config != "default":
            self.ctx.set_config(**AT.load(config)["config"])
        self.server = SV.Server(self.ctx, lanes=3, max_batch_views=64) if served else None

    def __del__(self):
        if getattr(self, "server", None) is not None:
            self.server.close()
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


_program = (None, None)


def _program_of(config, served):
    """The program of these settings: the latest one is kept, as a running
    program keeps its context."""
    global _program
    key = (config, served)
    if _program[0] != key:
        _program = (None, None)
        _program = (key, _Program(config, served))
    return _program[1]


class _State:
    """A program's resources for one case; closed in the order that their
    owners ask for."""

    def __init__(self, case, program):
        self.case, self.program, self.ctx = case, program, program.ctx
        self.closers = []

    def keep(self, x):
        self.closers.append(x)
        return x

    def __del__(self):
        for x in reversed(self.closers):
            x.close()


def _pinned(w, h, ids=False, depth=True):
    """Host buffers of a frame: colour, then depth and winner keys if read."""
    out = [torch.empty((h, w, 4), dtype=torch.uint8, pin_memory=True)]
    if depth:
        out.append(torch.empty((h, w), dtype=torch.float32, pin_memory=True))
    if ids:
        out.append(torch.empty((h, w), dtype=torch.int32, pin_memory=True))
    return out


def _pointers(bufs):
    kinds = (N._U8, N._F, N._U32)
    p = [C.cast(b.data_ptr(), k) for b, k in zip(bufs, kinds)]
    return p + [None] * (3 - len(p))


# ---- inputs ---------------------------------------------------------------------


def _sphere_faces(shape, faces):
    """(generator argument, faces, vertices) of a mesh of about `faces` faces."""
    if shape == "uv":
        k = max(4, int(round(math.sqrt(faces / 2.0))))
        return k, 2 * k * k, (k + 1) * (k + 1)
    n = max(2, int(round(math.sqrt(faces / 20.0))))
    return n, 20 * n * n, 10 * n * n + 2


def _object_sizes(case):
    """Face counts of a scene's objects, spread over its range."""
    m = case["objects"]
    lo, hi = math.log(case["faces_lo"]), math.log(case["faces_hi"])
    return [_sphere_faces(case["shape"], math.exp(lo + (hi - lo) * (i / (m - 1) if m > 1 else 1.0)))
            for i in range(m)]


def _log_sizes(lo, hi, m):
    return [math.exp(math.log(lo) + (math.log(hi) - math.log(lo)) * (i + 0.5) / m) for i in range(m)]


def _views_of(case):
    """(width, height) of a batch's views: 16:9 to square, over its range of heights."""
    out = []
    for i, s in enumerate(_log_sizes(case["s_lo"], case["s_hi"], case["views"])):
        h = int(s)
        out.append(((h, h * 4 // 3, h * 16 // 9)[i % 3], h))
    return out


def _requests_of(case):
    sizes = [(w, h) for w, h, _ in S.SERVE_RESOLUTIONS]
    pick = (0, 1, 0, 1, 0, 2, 0, 1, 0, 0)
    return [sizes[pick[i % 10]] for i in range(case["requests"])]


def _materials(st, case, rng, n):
    tex, filt = case["tex"], 1 if case.get("bilinear", True) else 0
    seed = lambda: int(rng.integers(1, 1 << 30))  # noqa: E731
    noise = lambda: st.keep(R.Texture(st.ctx, S.noise_texture(tex, tex, seed()), filt))  # noqa: E731
    normal = lambda: st.keep(R.Texture(st.ctx, S.normal_map(tex, tex, 0.7, seed()), filt))  # noqa: E731
    if case.get("shader") == "pbr":
        return [R.Material(noise(), noise(), normal(), noise(), noise(), 1.0) for _ in range(n)]
    return [R.Material(noise(), None, normal(), None, None, 0.64) for _ in range(n)]


def _shader(kind):
    sun = (0.3, -1.0, -0.4)
    return {"flat": R.FlatShader(lightDirection=sun), "phong": R.PhongShader(lightDirection=sun),
            "pbr": R.PBRShader(lightDirection=sun), "gouraud": R.GouraudShader(lightDirection=sun),
            "phong_point": R.PhongPointShader(lights=list(S.POINT_LIGHTS))}[kind]


def _camera(pos, w, h, target=(0.0, 0.0, 0.0)):
    cam = R.Camera(pos, target, 60.0, w / h)
    cam.setViewport(0, 0, w, h)
    cam.update(0.0)
    return cam


def _model(rng, spread, lo, hi):
    """Translation * rotation * scale, column-major."""
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    rot = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                    [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                    [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])
    m = np.eye(4)
    m[:3, :3] = rot * rng.uniform(lo, hi)
    m[:3, 3] = rng.uniform(-1.0, 1.0, 3) * spread
    return np.ascontiguousarray(m.T, dtype=np.float32).reshape(16)


def _prepare_scene(st, case, rng):
    ctx, w, h = st.ctx, case["width"], case["height"]
    mats = _materials(st, case, rng, case["groups"])
    st.draws = []
    one = case["objects"] == 1 and not case["close"]
    for arg, nf, _ in _object_sizes(case):
        if case["shape"] == "uv":
            v, f = S.uv_sphere(arg, arg)
            v[:, :3] *= (1.0 + 0.08 * rng.uniform(-1.0, 1.0, 3)).astype(np.float32)
        else:
            v, f = S.icosphere(arg, 0.1, int(rng.integers(1, 1 << 30)))
        cut = [nf * i // case["groups"] for i in range(case["groups"] + 1)]
        groups = [R.MaterialGroup(i, cut[i], cut[i + 1] - cut[i]) for i in range(case["groups"])]
        mesh = st.keep(R.Mesh(ctx, v, f, groups, mats))
        model = _model(rng, (0.05,) * 3 if one else (2.4, 1.4, 1.6), 0.9 if one else 0.45, 1.1 if one else 0.95)
        st.draws.append((model, mesh))
    # close: the camera stands among the objects, so some cross the planes
    yaw, pitch = rng.uniform(0.0, 360.0), rng.uniform(-20.0, 20.0)
    cam = _camera(S.orbit_position(3.0 if one else 1.3 if case["close"] else 4.6, yaw, pitch), w, h)
    st.fb = st.keep(R.Framebuffer(ctx, w, h, with_ids=case["ids"]))
    st.pipe = R.TiledPipeline(cam, st.fb)
    st.pipe.setShader(_shader(case["shader"]))
    st.out = _pinned(w, h, case["ids"])


def _prepare_frames(st, case, rng):
    ctx, w, h = st.ctx, case["width"], case["height"]
    v, f = S.icosphere(case["n"], 0.1, int(rng.integers(1, 1 << 30)))
    st.mesh = st.keep(R.Mesh(ctx, v, f, [R.MaterialGroup(0, 0, f.shape[0])], _materials(st, case, rng, 1)))
    st.fb = st.keep(R.Framebuffer(ctx, w, h))
    yaw, pitch = rng.uniform(0.0, 360.0), rng.uniform(-30.0, 30.0)
    model = np.eye(4, dtype=np.float32).reshape(16)
    st.params = [R.draw_params(model, _camera(S.orbit_position(3.0, yaw + 1.5 * i, pitch), w, h),
                               _shader("phong_point"), N.AXR_DRAW_ASYNC) for i in range(case["frames"])]
    st.out = _pinned(w, h)


def _prepare_soup(st, case, rng):
    ctx, w, h = st.ctx, case["width"], case["height"]
    v, f, c = S.soup(case["tris"], w, h, 60.0, 2.0, 1.5, 0.1, int(rng.integers(1, 1 << 30)))
    st.mesh = st.keep(R.Mesh(ctx, v, f, [R.MaterialGroup(0, 0, f.shape[0])], [R.Material()], c))
    st.fb = st.keep(R.Framebuffer(ctx, w, h))
    st.params = R.draw_params(np.eye(4, dtype=np.float32).reshape(16),
                              _camera((0.0, 0.0, 0.0), w, h, (0.0, 0.0, -1.0)), R.FlatColorShader())
    st.out = _pinned(w, h)


def _view_meshes(st, case, rng):
    mats = _materials(st, case, rng, 1)
    out = []
    for faces in _log_sizes(case["f_lo"], case["f_hi"], case["meshes"]):
        v, f = S.icosphere(_sphere_faces("ico", faces)[0], 0.1, int(rng.integers(1, 1 << 30)))
        out.append(st.keep(R.Mesh(st.ctx, v, f, [R.MaterialGroup(0, 0, f.shape[0])], mats)))
    return out


def _view_params(rng, w, h):
    pos = S.orbit_position(rng.uniform(2.2, 4.0), rng.uniform(0.0, 360.0), rng.uniform(-60.0, 60.0))
    return R.draw_params(np.eye(4, dtype=np.float32).reshape(16), _camera(pos, w, h), _shader("phong_point"))


def _prepare_batch(st, case, rng):
    meshes = _view_meshes(st, case, rng)
    sizes = _views_of(case)
    st.fbs = [st.keep(R.Framebuffer(st.ctx, w, h)) for w, h in sizes]
    st.batch = st.keep(R.Batch(st.ctx, st.fbs, [meshes[i % len(meshes)] for i in range(len(sizes))],
                               [_view_params(rng, w, h) for w, h in sizes]))
    st.batch.set_clear(RS.BLACK)
    st.out = [_pinned(w, h, depth=False)[0] for w, h in sizes]


def _prepare_serve(st, case, rng):
    meshes = _view_meshes(st, case, rng)
    sizes = _requests_of(case)
    st.requests = [(meshes[int(rng.integers(len(meshes)))], w, h, _view_params(rng, w, h)) for w, h in sizes]
    st.out = [_pinned(w, h, depth=False)[0] for w, h in sizes]


def prepare(case, seed):
    st = _State(case, _program_of(case["config"], case["kind"] == "serve"))
    rng = np.random.default_rng([int(seed), 77])
    {"scene": _prepare_scene, "frames": _prepare_frames, "soup": _prepare_soup, "batch": _prepare_batch,
     "serve": _prepare_serve}[case["kind"]](st, case, rng)
    return st


# ---- one pass ---------------------------------------------------------------------


def _complete(ctx, work):
    """Queue the work and wait for it, again while a frame arena reports that
    it had to grow (the frames since the last wait were then not drawn)."""
    for _ in range(8):
        work()
        try:
            ctx.sync()
            return
        except axr.AxrError as e:
            if e.code != N.AXR_ERR_OVERFLOW:
                raise
    raise RuntimeError("the frame arena kept overflowing")


def _read(st, fb, bufs):
    st.ctx.check(st.ctx._lib.axr_fb_read(fb.handle, *_pointers(bufs)))


def _run_scene(st):
    def frame():
        st.fb.clearColor(RS.BLACK)
        st.fb.clearDepth()
        for model, mesh in st.draws:
            st.pipe.drawMesh(model, mesh, asynchronous=st.case["queued"])

    if st.case["queued"]:
        _complete(st.ctx, frame)
    else:
        frame()
    _read(st, st.fb, st.out)


def _run_frames(st):
    lib, ctx, fb, mesh = st.ctx._lib, st.ctx, st.fb, st.mesh

    def frames():
        for p in st.params:
            lib.axr_fb_clear(fb.handle, RS.BLACK.packed_bgra(), float("inf"))
            ctx.check(lib.axr_draw(ctx.handle, fb.handle, mesh.handle, C.byref(p)))

    _complete(ctx, frames)
    _read(st, fb, st.out)


def _run_soup(st):
    lib, ctx = st.ctx._lib, st.ctx
    st.fb.clear(RS.BLACK)
    ctx.check(lib.axr_draw(ctx.handle, st.fb.handle, st.mesh.handle, C.byref(st.params)))
    _read(st, st.fb, st.out)


def _run_batch(st):
    _complete(st.ctx, st.batch.launch)
    for fb, out in zip(st.fbs, st.out):
        _read(st, fb, [out])


def _run_serve(st):
    srv = st.program.server
    tickets = [srv.submit(*q) for q in st.requests]
    for t, out in zip(tickets, st.out):
        srv.wait(t)
        srv.check(st.ctx._lib.axr_server_read(srv.handle, t, *_pointers([out])))
        srv.release(t)


def run(st):
    {"scene": _run_scene, "frames": _run_frames, "soup": _run_soup, "batch": _run_batch,
     "serve": _run_serve}[st.case["kind"]](st)
    return st.out


# ---- the work of one pass -----------------------------------------------------------


def _draw_work(nv, nf):
    """Positions and indices read once (12 bytes a vertex, 12 a face); the
    transform (28 operations a vertex) and the triangle setup (60 a face)."""
    return 12 * nv + 12 * nf, 28 * nv + 60 * nf


def work(case):
    """Bytes: positions and indices of every draw, colour and depth (and keys)
    of every finished frame, written once.  Operations: transform and setup;
    shading comes on top, by the pixels that a view happens to cover."""
    kind = case["kind"]
    draws, pixels = [], 0
    if kind == "scene":
        draws = [(nv, nf) for _, nf, nv in _object_sizes(case)]
        pixels = case["width"] * case["height"] * (12 if case["ids"] else 8)
    elif kind == "frames":
        n = case["n"]
        draws = [(10 * n * n + 2, 20 * n * n)] * case["frames"]
        pixels = case["width"] * case["height"] * 8 * case["frames"]
    elif kind == "soup":
        draws = [(3 * case["tris"], case["tris"])]
        pixels = case["width"] * case["height"] * 8
    else:
        sizes = _views_of(case) if kind == "batch" else _requests_of(case)
        meshes = [_sphere_faces("ico", f) for f in _log_sizes(case["f_lo"], case["f_hi"], case["meshes"])]
        draws = [(meshes[i % len(meshes)][2], meshes[i % len(meshes)][1]) for i in range(len(sizes))]
        pixels = 8 * sum(w * h for w, h in sizes)
    got = [_draw_work(nv, nf) for nv, nf in draws]
    return {"bytes": pixels + sum(b for b, _ in got), "flops": sum(f for _, f in got)}
