"""Spans that cross many tiles of one tile row: waves of them in tiles of one
and two pixels by 16 to 64, in windows of 64 tiles and over their ends.
Bit-exact against the oracle, and the span kernel's time over the rows."""
import numpy as np
import pytest

from conftest import announce
from test_gpu_blend_tiles import assert_both
import test_gpu_wide_waves as W

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


# columns 63 to 65 and 511 to 514 tiles from the first
@pytest.mark.parametrize("tiling", [(1, 64, 1), (1, 16, 2), (2, 64, 1)])
@pytest.mark.parametrize("width", [63, 64, 66, 515, 1031])
def test_windows(oracle, tiling, width):
    pos = np.concatenate([W.layers(2).reshape(-1, 3, 4), W.mixed(130, width, 75, width, hi=2.0 * width, every=3)])
    assert_both(W.scene(N.PROC_DEF03, pos, width, 75), oracle, tiling=tiling)


def test_span_time_over_rows():
    """tiles of 64 rows hold the same pieces as tiles of 16, of four times the
    spans of a wave: the span kernel takes up to 1.5 times as long, or, if each
    span looked through the others of its tile row, 3.2 times"""
    announce("span time over tile rows")
    sc = S.terrain_scene(1920, 1080, seed=5, tex_size=64)
    us = []
    for rows in (16, 64):
        with N.Context(sc.width, sc.height) as ctx:
            ctx.tiling(1, rows, 1)
            gs = S.GpuScene(ctx, sc)
            for _ in range(3):
                gs.frame()
            ctx.sync()
            ctx.profile(True)
            for _ in range(9):
                gs.frame()
            ms, launches = ctx.profile_read()["span"]
            us.append(ms / launches * 1e3)
    print(us)
    assert us[1] < 2.2 * us[0], us
