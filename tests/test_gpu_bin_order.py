"""The resolve of 16 and 32 px bins takes a workgroup per bin, in runs of four
neighbouring bins per XCD, rounded up to whole rounds of 32: bin counts around
those rounds, with a clear that the draw absorbs and without one."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("nx,ny", [(1, 1), (31, 1), (4, 8), (3, 11), (13, 5), (1, 129)])
def test_resolve_visits_every_bin_once(tile, nx, ny):
    sc = S.icosphere_scene(n=6, width=nx * tile - 3, height=ny * tile - 1, tex=64, radius=2.2)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=N.RASTER_VISIBILITY, tile_size=tile)
        gs = H.GpuScene(ctx, sc)
        fbs = [R.Framebuffer(ctx, sc.width, sc.height, with_ids=True) for _ in range(2)]
        try:
            p = H.params_of(sc)
            for k, fb in enumerate(fbs):
                fb.clear(R.Color(1, 2, 3, 4), 0.1)
                fb.read()                       # settles that clear
                fb.clear(R.Color(7, 77, 177, 3))
                if k == 1:
                    fb.read()                   # the clear as a pass of its own
                for _ in range(2):
                    ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, R.C.byref(p)))
            a, b = fbs[0].read(), fbs[1].read()
            for x, y in zip(a, b):
                assert (x.view(np.uint8) == y.view(np.uint8)).all()
        finally:
            for fb in fbs:
                fb.close()
            gs.close()
        rep = H.compare(H.render_gpu(ctx, sc), H.render_oracle(sc))
        H.assert_parity(rep, f"{nx} x {ny} bins of {tile}")
        assert rep["covered"] > 0
    finally:
        ctx.close()
