"""Tiles of chunks of 16 to 64 pixels, whose pieces each lane walks for its own
chunk: hundreds of triangles on a few tiles, spans of up to several chunks and
of a pixel, draws that test and update depth in every combination, widths and
heights that end within a chunk and a tile.  Bit-exact against the oracle, with
and without the debug planes, and the raster kernel's time over the width."""
import pytest

from conftest import announce
from test_gpu_blend_tiles import assert_both, crowded_layers
from test_gpu_tile_lists import crowded_scene
import test_gpu_wide_waves as W

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402

TILINGS = [(16, 1, 2), (16, 16, 3), (16, 64, 1), (32, 4, 2), (32, 64, 1), (64, 1, 1), (64, 8, 1), (64, 64, 1)]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("tiling", TILINGS)
def test_crowded(oracle, tiling, mixed):
    assert_both(crowded_scene(900, 175, 71, 23, mixed), oracle, tiling=tiling)


@pytest.mark.parametrize("prog", [N.PROC_CLOUD, N.PROC_CLOUD_SHADOW])
@pytest.mark.parametrize("tiling", TILINGS)
def test_crowded_layers(oracle, tiling, prog):
    assert_both(crowded_layers(prog, 260, 175, 71, 29, True), oracle, tiling=tiling)


@pytest.mark.parametrize("tiling", [(16, 16, 1), (32, 8, 1), (64, 32, 1)])
def test_layers_across(oracle, tiling):
    assert_both(W.scene(N.PROC_DEF03, W.layers(70), 259, 70), oracle, tiling=tiling)


def raster_us(sc, tiling):
    with N.Context(sc.width, sc.height) as ctx:
        ctx.tiling(*tiling)
        gs = S.GpuScene(ctx, sc)
        for _ in range(3):
            gs.frame()
        ctx.sync()
        ctx.profile(True)
        for _ in range(9):
            gs.frame()
        ms, launches = ctx.profile_read()["raster"]
        return ms / launches * 1e3


def test_raster_time_over_chunks():
    """chunks of 64 pixels leave a tile's wave with four times the pixels of
    chunks of 16: the walk takes about twice as long, or as it went through all
    64 pixels of the chunk in turn 3.5 times; of a blended layer, the tiles 16
    and 64 rows high, 4.4 and 6.5 times"""
    announce("raster time over chunk widths")
    opaque = S.terrain_scene(1920, 1080, seed=5, tex_size=64)
    got = [raster_us(opaque, t) for t in ((16, 8, 1), (64, 4, 1))]
    blended = S.cloud_terrain_scene(960, 540, seed=5, tex_size=64)
    got += [raster_us(blended, t) for t in ((16, 16, 1), (64, 64, 1))]
    print(got)
    assert got[1] < 2.7 * got[0] and got[3] < 5.9 * got[2], got
