"""Binned mode's bins: entries written straight into a bin's first level and,
past it, into levels from the pools (raster.hip bin_put / bin_get), by the
wave's rounds (grouped or lane by lane) and by its flattened pairs; and the
wave-per-face clipper that feeds them.  Every frame equals the oracle's,
bit for bit in coverage, depth and winner."""
import numpy as np
import pytest

import harness as H
from axiomr_amd import _native as N
from axiomr_amd import render as R
from axiomr_amd import scenes as S


def _scene(kind):
    if kind == "clustered":     # 81,920 faces in a few bins: several levels past the first
        return S.icosphere_scene(n=64, width=640, height=480, tex=64, radius=45.0)
    if kind == "one_bin":       # a window no larger than a bin
        return S.icosphere_scene(n=32, width=7, height=5, tex=64)
    if kind == "large":         # triangles over most of the bins, odd size
        return S.icosphere_scene(n=2, width=1283, height=719, tex=64)
    if kind == "inside":        # the camera below the surface: clipped faces, none of them facing it
        return S.icosphere_scene(n=9, width=333, height=251, tex=64, radius=1.03)
    if kind == "clipped":       # faces across the screen's edges and corners
        return S.icosphere_scene(n=9, width=333, height=251, tex=64, radius=1.3)
    return S.soup_scene(ntri=30_001, width=321, height=203, seed=12)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("kind", ["clustered", "one_bin", "large", "inside", "clipped", "soup"])
def test_bins_equal_oracle(kind, tile):
    sc = _scene(kind)
    ref = H.render_oracle(sc)
    ctx = R.Context(0)
    try:
        ctx.set_config(raster_mode=N.RASTER_BINNED, tile_size=tile)
        for again in range(2):          # the second frame runs on an arena the first one cleaned
            rep = H.compare(H.render_gpu(ctx, sc), ref)
            H.assert_parity(rep, f"{kind} tile {tile} frame {again}")
        assert (rep["covered"] > 0) == (kind != "inside")
    finally:
        ctx.close()


def test_levels_cover_every_slot_once():
    """level(s) = 31 - clz((s >> shift) + 1) and its offset, as bin_slot
    computes them: consecutive slots fill each level in turn, none twice."""
    for shift in (5, 9, 12):
        s = np.arange(0, 1 << 18, dtype=np.uint64)
        q = (s >> np.uint64(shift)) + np.uint64(1)
        level = np.floor(np.log2(q.astype(np.float64))).astype(np.uint64)
        offset = s - (((np.uint64(1) << level) - np.uint64(1)) << np.uint64(shift))
        size = np.uint64(1) << (np.uint64(shift) + level)
        assert (offset < size).all()
        first = np.flatnonzero(offset == 0)
        assert (np.diff(level[first]) == 1).all() and level[0] == 0
        assert (np.diff(s)[np.diff(level) == 0] == 1).all()


def test_count_words_are_a_permutation_of_each_block():
    """count_word as the kernels compute it: every block of 8,192 bins maps
    onto itself one to one, runs of four bins stay together, and neighbouring
    runs lie in different 128-byte lines."""
    t = np.arange(3 * 8192, dtype=np.int64)
    w = (t & ~8191) | ((t & 0x3FC) << 3) | (t & 3) | ((t >> 8) & 28)
    assert (np.sort(w) == t).all() and (w >> 13 == t >> 13).all()
    assert (w[1::4] == w[0::4] + 1).all() and (w[3::4] == w[0::4] + 3).all()
    line = w[0::4] >> 5
    assert (line[1:] != line[:-1]).all()
