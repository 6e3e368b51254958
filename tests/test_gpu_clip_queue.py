"""The clipper's queue: faces within the sub-queues, past them into the shared
queue, and past that (the arena grows and the frame is drawn again), one to
several pieces a face; every frame equals the oracle's."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S

pytestmark = pytest.mark.gpu


def edge_scene(n, corner, seed=8, width=403, height=301):
    """n small front-facing triangles across the left frustum plane or, with
    `corner`, around the lower left corner (two planes, up to three pieces)."""
    rng = np.random.default_rng(seed)
    t = np.tan(np.radians(30.0))
    z = rng.uniform(1.0, 20.0, n)
    cx = -z * t * width / height
    cy = -z * t if corner else rng.uniform(-0.95, 0.95, n) * z * t
    size = z * rng.uniform(0.01, 0.08, n)
    a = rng.uniform(0, 2 * np.pi, n)
    v = np.zeros((n, 3, 14), np.float32)
    for k in range(3):
        v[:, k, 0] = cx + size * np.cos(a + k * 2 * np.pi / 3)
        v[:, k, 1] = cy + size * np.sin(a + k * 2 * np.pi / 3)
        v[:, k, 2] = -z
    v[:, :, 5:8] = (0.0, 0.0, 1.0)
    f = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    colors = rng.integers(0, 2**32, n, dtype=np.uint64).astype(np.uint32)
    return S.SceneData(name=f"edge_{n}", vertices=v.reshape(-1, 14), faces=f, width=width, height=height,
                       camera_pos=(0.0, 0.0, 0.0), camera_target=(0.0, 0.0, -1.0), fov=60.0, shader={"kind": 5},
                       groups=[(0, 0, n)], materials=[S.MaterialData()], face_colors=colors)


@pytest.mark.parametrize("mode", [N.RASTER_BINNED, N.RASTER_VISIBILITY])
@pytest.mark.parametrize("n,corner", [(65, False), (3000, False), (3000, True), (7000, False), (20_000, True)])
def test_clip_queue_equals_oracle(mode, n, corner):
    sc = edge_scene(n, corner)
    ref = H.render_oracle(sc)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=mode, small_footprint=64)
        for again in range(2):
            rep = H.compare(H.render_gpu(ctx, sc), ref)
            H.assert_parity(rep, f"{n} corner {corner} frame {again}")
        assert rep["covered"] > 50
    finally:
        ctx.close()
