"""More bins than one launch holds a workgroup each for: a batch of thin, tall
views whose bins pass 2^23, views on both sides of that line equal to their
solo draws."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu

HEIGHT, VIEWS = 32768, 4100      # 2,048 bins of 16 px each: view 4,096 starts the second launch
SEEN = (0, 4095, 4096, 4099)


@pytest.mark.parametrize("mode", [N.RASTER_BINNED, N.RASTER_VISIBILITY])
def test_bins_over_one_launch(mode):
    sc = S.icosphere_scene(n=2, width=2, height=HEIGHT, tex=16, radius=2.3)
    see, away = H.params_of(sc), H.params_of(sc)
    model = np.eye(4, dtype=np.float32)
    model[3, :3] = 3.0 * np.array(sc.camera_pos, np.float32)     # behind the camera
    away.model[:] = [float(x) for x in model.reshape(16)]
    ctx = R.Context(0)
    fbs, batch, gs = [], None, None
    try:
        ctx.set_config(raster_mode=mode, tile_size=16)
        gs = H.GpuScene(ctx, sc)
        fbs = [R.Framebuffer(ctx, 2, HEIGHT) for _ in range(VIEWS)]
        batch = R.Batch(ctx, fbs, [gs.mesh] * VIEWS, [see if i in SEEN else away for i in range(VIEWS)])
        batch.set_clear(R.Color(9, 8, 7, 6))
        for _ in range(4):      # an overflow is reported, with the arena grown for the next launch
            batch.launch()
            try:
                ctx.sync()
                break
            except N.AxrError as e:
                assert e.code == N.AXR_ERR_OVERFLOW
        else:
            pytest.fail("kept overflowing")
        got = {i: fbs[i].read() for i in SEEN + (1, 4098)}
        fbs[0].clear(R.Color(9, 8, 7, 6))
        ctx.check(ctx._lib.axr_draw(ctx.handle, fbs[0].handle, gs.mesh.handle, R.C.byref(see)))
        want = fbs[0].read()
        assert np.isfinite(want[1]).sum() > 1000
        for i in SEEN:
            for a, b in zip(got[i][:2], want[:2]):
                assert (a.view(np.uint8) == b.view(np.uint8)).all(), f"view {i}"
        for i in (1, 4098):
            assert np.isinf(got[i][1]).all(), f"view {i}"
    finally:
        if batch:
            batch.close()
        for fb in fbs:
            fb.close()
        if gs:
            gs.close()
        ctx.close()
