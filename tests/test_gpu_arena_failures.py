"""Frame arenas after a growth that an HBM budget refused, at every buffer
the growth may stop at: the draw that needed it reports the budget, and the
frames after it, in either raster mode, have the oracle's pixels."""
import pytest

import axiomr_amd as axr
import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu

MODES = [N.RASTER_BINNED, N.RASTER_VISIBILITY]
SPARE = 4 << 20       # bytes given back after the refused draw, for the frames that follow


class Frame:
    def __init__(self, ctx, sc):
        self.ctx, self.gs = ctx, H.GpuScene(ctx, sc)
        self.fb = R.Framebuffer(ctx, sc.width, sc.height, with_ids=True)
        self.params = H.params_of(sc)

    def draw(self, mode):
        self.ctx.set_config(raster_mode=mode, tile_size=8)
        self.fb.clear(H.BLACK)
        self.ctx.check(self.ctx._lib.axr_draw(self.ctx.handle, self.fb.handle, self.gs.mesh.handle, R.C.byref(self.params)))

    def close(self):
        self.fb.close()
        self.gs.close()


@pytest.mark.parametrize("refused", MODES)
@pytest.mark.parametrize("after", [(m,) for m in MODES] + [(MODES[0], MODES[1]), (MODES[1], MODES[0])])
def test_frames_after_a_refused_growth(refused, after):
    large = S.icosphere_scene(n=20, width=1600, height=1200, tex=64)
    small = [S.icosphere_scene(n=12, width=w, height=64, tex=64) for w in (64, 96)]
    refs = [H.render_oracle(sc) for sc in small]

    def run(budget, refuse):
        """The large draw in a context with `budget` bytes: refused, with the
        frames after it, or (not `refuse`) drawn; the bytes in use before it
        and those that its arena takes beyond the small frames'."""
        ctx = R.Context(0, budget)
        open_ = []
        try:
            first, big, last = [open_.append(Frame(ctx, sc)) or open_[-1] for sc in (small[0], large, small[1])]
            spare = R.Framebuffer(ctx, 1024, SPARE // 8 // 1024)
            open_.append(spare)
            for mode in MODES:
                first.draw(mode)
            used, arena = ctx.memory()
            if not refuse:
                big.draw(refused)
                return used + arena, ctx.memory()[1] - arena
            with pytest.raises(axr.AxrError) as e:
                big.draw(refused)
            assert e.value.code == N.AXR_ERR_BUDGET
            open_.pop().close()
            for again in range(2):
                for mode in after:
                    for frame, ref in ((first, refs[0]), (last, refs[1])):
                        frame.draw(mode)
                        H.assert_parity(H.compare(frame.fb.read(), ref), f"budget {budget} mode {mode} frame {again}")
        finally:
            for x in reversed(open_):
                x.close()
            ctx.close()

    base, growth = run(8 << 30, refuse=False)
    assert growth > 1 << 20
    for eighth in range(8):
        print(f"refused {refused} after {after}: {eighth}/8 of {growth} bytes", flush=True)
        run(base + growth * eighth // 8, refuse=True)
