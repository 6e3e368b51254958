"""Read-backs: into pinned buffers (one launch for all planes, or a runtime
copy for a single one), into ordinary memory, at sizes whose planes end
inside a 16-byte store, and into pinned memory at offsets that such stores
cannot take: always the same bytes."""
import ctypes as C

import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu


class Pinned:
    """Pinned host memory from the HIP runtime that the library runs on,
    filled with a pattern; .array is the whole block, .address word `offset`."""

    def __init__(self, words, offset):
        self.hip = C.CDLL("libamdhip64.so.7")
        p = C.c_void_p()
        total = words + offset + 8
        assert self.hip.hipHostMalloc(C.byref(p), C.c_size_t(4 * total), C.c_uint(0)) == 0
        self.base = p.value
        self.array = np.frombuffer((C.c_uint32 * total).from_address(self.base), np.uint32)
        self.array[:] = 0x5A5A5A5A
        self.address = self.base + 4 * offset

    def close(self):
        self.array = None
        assert self.hip.hipHostFree(C.c_void_p(self.base)) == 0


@pytest.mark.parametrize("width,height", [(1, 1), (5, 3), (64, 64), (333, 217), (1920, 1080)])
@pytest.mark.parametrize("offset", [0, 4, 1])
def test_pinned_reads_equal_plain_reads(ctx, width, height, offset):
    sc = S.icosphere_scene(n=12, width=width, height=height, tex=64)
    gs = H.GpuScene(ctx, sc)
    fb = R.Framebuffer(ctx, width, height, with_ids=True)
    try:
        n = width * height
        for flags in (0, N.AXR_DRAW_ASYNC):      # an asynchronous draw is waited for by the read itself
            fb.clear(R.Color(3, 4, 5, 6))
            p = H.params_of(sc, flags=flags)
            ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, C.byref(p)))
            for planes in ((1, 1, 1), (1, 1, 0), (0, 1, 1), (1, 0, 0)):
                bufs = [Pinned(n, offset) if on else None for on in planes]
                ptrs = [C.cast(b.address, k) if b else None for b, k in zip(bufs, (N._U8, N._F, N._U32))]
                ctx.check(ctx._lib.axr_fb_read(fb.handle, *ptrs))
                plain = [x.view(np.uint32).reshape(-1) for x in fb.read()]
                for b, want in zip(bufs, plain):
                    if b is None:
                        continue
                    got = b.array.copy()
                    b.close()
                    assert (got[offset:offset + n] == want).all()
                    assert (got[:offset] == 0x5A5A5A5A).all() and (got[offset + n:] == 0x5A5A5A5A).all()
        ctx.sync()
    finally:
        fb.close()
        gs.close()


def test_waits_longer_than_the_poll():
    """A synchronous draw and an axr_sync behind several milliseconds of
    queued work, which outlast the polled part of the wait."""
    ctx = R.Context(0)
    try:
        sc = S.soup_scene(ntri=1_500_000, width=1024, height=768, seed=5)
        gs = H.GpuScene(ctx, sc)
        fb = R.Framebuffer(ctx, sc.width, sc.height, with_ids=True)
        fb.clear(H.BLACK)
        p, q = H.params_of(sc), H.params_of(sc, flags=N.AXR_DRAW_ASYNC)
        ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, C.byref(p)))
        want = fb.read()
        for last in (p, q):
            fb.clear(H.BLACK)
            for _ in range(25):
                ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, C.byref(q)))
            ctx.check(ctx._lib.axr_draw(ctx.handle, fb.handle, gs.mesh.handle, C.byref(last)))
            ctx.sync()
            for a, b in zip(fb.read(), want):
                assert (a.view(np.uint8) == b.view(np.uint8)).all()
        fb.close()
        gs.close()
    finally:
        ctx.close()
