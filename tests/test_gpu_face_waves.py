"""Passes over faces by their launch rules: 16 or 64 faces per wave, walks of
larger rectangles shared by the wave or not (k_vis), bin entries laid end to
end, workgroup sizes of the binned raster, and clears absorbed by it.  Every
frame equals the oracle's; batched views whose faces share a wave equal
their solo draws."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu

MODES = {"binned": N.RASTER_BINNED, "visibility": N.RASTER_VISIBILITY}


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n,width,height,footprint", [
    (1, 129, 97, 1024),         # 20 faces: one full wave of 16 and a rest
    (4, 801, 603, 1024),        # rectangles of hundreds of pixels, shared
    (40, 1280, 720, 128),       # 32,000 faces: the last count of 16 per wave
    (41, 1280, 720, 12),        # 33,620: 64 per wave, shared
    (41, 640, 480, 128),        # 9 pixels per face: not shared
])
def test_face_waves_equal_oracle(mode, n, width, height, footprint):
    sc = S.icosphere_scene(n=n, width=width, height=height, tex=64, radius=2.3)
    ref = H.render_oracle(sc)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=MODES[mode], small_footprint=footprint)
        rep = H.compare(H.render_gpu(ctx, sc), ref)
        H.assert_parity(rep, f"{mode} n {n}")
        assert rep["covered"] > 1000
    finally:
        ctx.close()


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("tile", [8, 16, 32])
def test_batch_views_sharing_a_wave(mode, tile):
    """Views of 20 and 80 faces at sizes that share walks: most waves hold
    faces of two views, of different sizes and with different bins."""
    wl = S.batch_workload(nviews=7, nmeshes=2, fmin=20, fmax=81, wmin=60, wmax=500, hmin=50, hmax=400, tex=64, seed=3)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=MODES[mode], tile_size=tile, small_footprint=1024)
        gb = H.GpuBatch(ctx, wl)
        try:
            gb.batch.launch()
            ctx.sync()
            batched = [fb.read() for fb in gb.fbs]
            for i in range(len(wl.views)):
                gb.draw_solo(i)
                for a, b in zip(batched[i], gb.fbs[i].read()):
                    assert (a.view(np.uint8) == b.view(np.uint8)).all(), f"view {i}"
            H.assert_parity(H.compare(batched[0], H.render_oracle(wl.scene(0))), "view 0")
        finally:
            gb.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("depth", [float("inf"), 0.9])
def test_binned_clear_in_the_raster(tile, threads, depth):
    """A binned draw writes the clear it absorbs over every pixel of an odd
    target, winners behind the clear depth included; a second draw without a
    clear keeps what is there."""
    sc = S.icosphere_scene(n=8, width=203, height=101, tex=64)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=N.RASTER_BINNED, tile_size=tile, raster_threads=threads)
        gs = H.GpuScene(ctx, sc)
        fbs = [R.Framebuffer(ctx, sc.width, sc.height, with_ids=True) for _ in range(2)]
        try:
            p = H.params_of(sc)
            tint = R.Color(7, 77, 177, 3)
            for k, fb in enumerate(fbs):
                fb.clear(R.Color(1, 2, 3, 4), 0.1)
                fb.read()                       # settles that clear
                fb.clear(tint, depth)
                if k == 1:
                    fb.read()                   # the clear as a pass of its own
                for _ in range(2):
                    ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, R.C.byref(p)))
            a, b = fbs[0].read(), fbs[1].read()
            for x, y in zip(a, b):
                assert (x.view(np.uint8) == y.view(np.uint8)).all()
            assert (a[2] == 0xFFFFFFFF).sum() > 1000
        finally:
            for fb in fbs:
                fb.close()
            gs.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("counts", [(700, 0, 580), (1, 638, 0, 641), (3, 5, 7, 11, 1254), (0, 0, 1280)])
def test_material_groups(mode, counts):
    """Two to five groups (up to four are searched without loads), empty ones
    among them, submitted in another order than the index buffer's, with a
    material each."""
    base = S.icosphere_scene(n=8, width=320, height=240, tex=64)
    first = np.cumsum((0,) + counts[:-1])
    order = list(range(len(counts)))[::-1]
    mats, tex = [], dict(base.textures)
    for i in range(len(counts)):
        tex[f"albedo{i}"] = S.TextureData(S.noise_texture(32, 32, 50 + i), i % 2)
        mats.append(S.MaterialData(diffuse=f"albedo{i}", bump="normal", specular_exponent=0.3 + 0.2 * i))
    sc = S.with_shader(base, base.shader, materials=mats, textures=tex)
    sc.groups = [(i, int(first[i]), int(counts[i])) for i in order]
    assert sum(counts) == sc.nfaces
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=MODES[mode])
        ref = H.render_oracle(sc)
        rep = H.compare(H.render_gpu(ctx, sc), ref)
        H.assert_parity(rep, f"{mode} groups {counts}")
        assert rep["covered"] > 1000
    finally:
        ctx.close()
