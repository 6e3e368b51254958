"""Frame arenas that an HBM budget counts: no larger than arenas that kept
their bins as sorted pairs (28 bytes a face and 332 a bin beside the records
and the clipper's room), which budgets were chosen for, with the same pixels
as arenas without a budget."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu


def pair_arena_bytes(faces, bins, capacity=64):
    """An arena with one region of `capacity` 16-byte pairs per 64 faces."""
    faces, bins = max(faces, 1024), max(bins, 1024)     # every arena starts with room for these
    clip = max(4096, faces // 16)
    waves = 4 * ((faces + 255) // 256)
    pairs = 16 * (waves * capacity + faces // 4 + 16 * bins + 4096) + 4 * waves
    entries = 4 * (2 * faces + 16 * bins + 4096)
    return 48 * faces + clip * (4 + 2 * (48 + 168)) + pairs + entries + 12 * (bins + 1)


def draw(sc, budget, tile):
    ctx = R.Context(0, budget)
    try:
        ctx.set_config(raster_mode=N.RASTER_BINNED, tile_size=tile)
        gs = H.GpuScene(ctx, sc)
        fb = R.Framebuffer(ctx, sc.width, sc.height, with_ids=True)
        try:
            p = H.params_of(sc)
            fb.clear(R.Color(0, 0, 0, 255))
            ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, R.C.byref(p)))
            return fb.read(), ctx.memory()[1]
        finally:
            fb.close()
            gs.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("kind,n,width,height,tile", [
    ("mesh", 2, 64, 64, 8),             # 80 faces
    ("mesh", 4, 1920, 1080, 8),         # 320 faces over 32,400 bins
    ("mesh", 60, 640, 360, 32),         # 72,000 faces over 240 bins
    ("soup", 60_000, 320, 200, 16),     # bins of many levels
    ("inside", 60, 500, 300, 16),       # the camera inside: clipped faces, all seen from behind
    ("near", 60, 500, 300, 16),         # just outside: clipped faces seen from the front
])
def test_budgeted_arena(kind, n, width, height, tile):
    if kind == "soup":
        sc = S.soup_scene(n, width, height)
    else:
        sc = S.icosphere_scene(n=n, width=width, height=height, tex=64, radius={"inside": 0.5, "near": 1.15, "mesh": 2.3}[kind])
    want, _ = draw(sc, 0, tile)
    got, arena = draw(sc, 8 << 30, tile)
    for a, b in zip(got, want):
        assert (a.view(np.uint8) == b.view(np.uint8)).all()
    if kind == "mesh":      # the others grow by what their first try reports
        faces = 20 * n * n
        assert arena <= pair_arena_bytes(faces, ((width + tile - 1) // tile) * ((height + tile - 1) // tile))
    assert kind == "inside" or (got[2] != 0xFFFFFFFF).sum() > 100
