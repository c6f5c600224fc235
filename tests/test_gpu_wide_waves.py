"""Waves of span items that hold a wide span: their pieces of a tile are one
run, whichever waves place the spans.  Waves across more tiles than the span
kernel's bins, tile rows that one wave meets in several triangles, tile rows of
one to 64 rows, many columns and few, several views, scratch that starts tiny
and flushes that are split.  Bit-exact against the oracle, with and without the
debug planes, and the raster kernel's time over the number of layers."""
import numpy as np
import pytest

from conftest import announce
import scenegen
from test_gpu_blend_tiles import assert_both

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


def scene(prog, pos, width, height, seed=3):
    sc = scenegen.micro_scene(prog, seed, width, height, n=24)
    sc.meshes["m"] = scenegen._slots_for(prog, pos.reshape(-1, 4).astype(np.float32), np.random.default_rng(seed))
    sc.draws = sc.draws[:1]
    sc.draws[0].behavior = N.UPDATE_DEPTH | N.TEST_DEPTH
    sc.name = "wide_waves_p%d_%d_%dx%d" % (prog, len(pos.reshape(-1, 3, 4)), width, height)
    return sc


def layers(n):
    """n pairs of triangles across the view, each nearer than the one before"""
    q = np.zeros((n, 2, 3, 4))
    c = np.array([(-1, -1), (1, -1), (1, 1), (-1, 1)], float)
    q[:, 0, :, :2], q[:, 1, :, :2] = c[[0, 1, 2]], c[[0, 2, 3]]
    q[..., 2] = np.linspace(0.9, -0.9, n)[:, None, None]
    q[..., 3] = 1.0
    return q


def mixed(n, width, height, seed, lo=3.0, hi=90.0, every=4):
    """n triangles of a few pixels, each `every`-th of up to hi, anywhere"""
    r = np.random.default_rng(seed)
    size = r.uniform(lo, lo + 6, n)
    size[::every] = r.uniform(hi / 2, hi, len(size[::every]))
    a = r.uniform(0, 2 * np.pi, n)[:, None] + np.arange(3) * 2 * np.pi / 3
    p = np.ones((n, 3, 4))
    p[..., 0] = r.uniform(-1, 1, (n, 1)) + np.cos(a) * size[:, None] / width
    p[..., 1] = r.uniform(-1, 1, (n, 1)) + np.sin(a) * size[:, None] / height
    p[..., 2] = r.uniform(-0.9, 0.9, (n, 1))
    return p


# a wave across a 1080p screen meets 540 tiles, 60 of them in a row
@pytest.mark.parametrize("prog", [N.PROC_DEF02, N.PROC_DEF05])
def test_across_the_screen(oracle, prog):
    assert_both(scene(prog, np.concatenate([layers(2).reshape(-1, 3, 4), mixed(40, 1920, 1080, 1, hi=700.0)]), 1920, 1080), oracle)


@pytest.mark.parametrize("prog", [N.PROC_DEF02, N.PROC_DEF03, N.PROC_DEF05, N.PROC_BLINN, N.PROC_CLOUD])
@pytest.mark.parametrize("every", [2, 9])
def test_among_small_triangles(oracle, prog, every):
    assert_both(scene(prog, mixed(900, 518, 301, 7 + prog, every=every), 518, 301), oracle)


@pytest.mark.parametrize("tiling", [(1, 8, 2), (1, 64, 1), (2, 1, 4), (4, 16, 2), (8, 64, 3), (16, 4, 1), (64, 2, 1)])
def test_tilings(oracle, tiling):
    assert_both(scene(N.PROC_DEF03, mixed(500, 411, 133, 5, hi=250.0), 411, 133), oracle, tiling=tiling)


# as many runs a tile as layers: in the lanes, in LDS and in memory
@pytest.mark.parametrize("n", [63, 65, 255, 259])
def test_layers(oracle, n):
    assert_both(scene(N.PROC_DEF02, layers(n), 102, 23), oracle)


# PSGPU_CREATE_TINY_SCRATCH and PSGPU_CREATE_SMALL_FLUSHES
@pytest.mark.parametrize("flags,seen", [(1, "retries"), (2, "splits")])
def test_scratch_limits(oracle, flags, seen):
    sc = scene(N.PROC_DEF02, np.concatenate([mixed(300, 158, 87, 11), layers(2).reshape(-1, 3, 4)]), 158, 87)
    announce("%s flags %d" % (sc.name, flags))
    f, ost = oracle.render_scene(sc)
    with N.Context(sc.width, sc.height, flags=flags) as ctx:
        gs = S.GpuScene(ctx, sc)
        for _ in range(2):
            gs.frame()
            np.testing.assert_array_equal(ctx.read_depth().view(np.uint32), f.depth.view(np.uint32))
            np.testing.assert_array_equal(ctx.read_colour(), f.colour)
        st = ctx.stats()
        assert st[seen] > 0
        assert st["frags_shaded"] == 2 * ost.frags_shaded


def test_several_views():
    """views of one flush against the views rendered one by one"""
    sc = scene(N.PROC_DEF03, np.concatenate([mixed(200, 230, 90, 2), layers(3).reshape(-1, 3, 4)]), 230, 90)
    announce(sc.name + " in three views")
    with N.Context(sc.width, sc.height) as ctx:
        gs = S.GpuScene(ctx, sc)
        images = []
        for together in (False, True):
            views = [(w, h, ctx.texture_create(w, h, 4, wrap=N.CLAMP), ctx.texture_create(w, h, 4, wrap=N.CLAMP))
                     for w, h in ((230, 90), (77, 41), (120, 8))]
            for w, h, c, d in views:
                ctx.target(c)
                ctx.depth_target(d)
                ctx.viewport(w, h)
                ctx.clear_depth(1.0)
                ctx.clear_target(7)
                gs.frame(clear=False, flush=not together)
            flushes = ctx.stats()["flushes"]
            ctx.sync()
            assert not together or ctx.stats()["flushes"] == flushes + 1
            images.append([ctx.texture_download(t).ravel() for v in views for t in v[2:]])
    for a, b in zip(*images):
        np.testing.assert_array_equal(a, b)


def test_raster_time_over_layers():
    """48 layers hold twice the pieces of 24, and tiles of 48 and 24 runs: the
    raster kernel takes about twice as long, not seven times (tiles of eight
    runs a layer, beyond what is sorted in LDS, took 7.5 times)"""
    announce("raster time over layers")
    us = []
    for n in (24, 48):
        sc = scene(N.PROC_DEF02, layers(n), 1920, 1080)
        with N.Context(sc.width, sc.height) as ctx:
            gs = S.GpuScene(ctx, sc)
            for _ in range(3):
                gs.frame()
            ctx.sync()
            ctx.profile(True)
            for _ in range(9):
                gs.frame()
            ms, launches = ctx.profile_read()["raster"]
            us.append(ms / launches)
    assert us[1] < 4.0 * us[0], us
