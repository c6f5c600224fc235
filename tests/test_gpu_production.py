"""The kernels of an ordinary context, without debug planes, which are their own
instances: the scenes of the tile lists, the wide spans and the draws, every
chunk width, several waves a group, and replays of a captured frame.  Bit-exact
against the oracle."""
import numpy as np
import pytest

from conftest import announce
from test_gpu_parity import gpu_render
from test_gpu_shade_draws import PROGS, draws_scene, programmes_scene
from test_gpu_tile_lists import crowded_scene
from test_gpu_wide_spans import wide_scene

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402

TILINGS = [(1, 8, 8), (2, 16, 1), (4, 8, 2), (8, 8, 8), (8, 64, 3), (16, 4, 5), (32, 2, 3), (64, 1, 1)]


def assert_production(sc, oracle, tiling=None):
    announce("%s %s" % (sc.name, tiling))
    col, dep, _, st = gpu_render(sc, tiling, debug=False)
    f, ost = oracle.render_scene(sc)
    np.testing.assert_array_equal(dep.view(np.uint32), f.depth.view(np.uint32))
    np.testing.assert_array_equal(col, f.colour)
    assert st["frags_shaded"] == ost.frags_shaded


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [40, 700, 820, 840, 3000, 5000])
def test_crowded_tile(oracle, n, mixed):
    assert_production(crowded_scene(n, 31, 8, n, mixed), oracle)


@pytest.mark.parametrize("tiling", TILINGS)
def test_crowded_tilings(oracle, tiling):
    assert_production(crowded_scene(1500, 47, 35, 5, True), oracle, tiling)


@pytest.mark.parametrize("prog", [N.PROC_DEF03, N.PROC_DEF05, N.PROC_LAMBERT, N.PROC_BLINN])
@pytest.mark.parametrize("lengths", [False, True])
def test_wide_spans(oracle, prog, lengths):
    assert_production(wide_scene(prog, 40, 1507, 37, 3 + prog, lengths), oracle)


@pytest.mark.parametrize("tiling", TILINGS)
def test_wide_span_tilings(oracle, tiling):
    assert_production(wide_scene(N.PROC_BLINN, 30, 1102, 70, 9), oracle, tiling)


@pytest.mark.parametrize("n_draws", [1, 9])
@pytest.mark.parametrize("prog", PROGS)
def test_draws_of_a_programme(oracle, prog, n_draws):
    assert_production(draws_scene(prog, n_draws, 40 + prog, 47, 35), oracle)


def test_programmes_of_one_flush(oracle):
    assert_production(programmes_scene(94, 131, 37, PROGS[::-1] + PROGS * 2), oracle)


def test_captured_frame(oracle):
    """replays of one graph, with eager frames between them"""
    sc = crowded_scene(700, 131, 35, 3, True)
    announce("captured " + sc.name)
    f, _ = oracle.render_scene(sc)
    with N.Context(sc.width, sc.height) as ctx:
        gs = S.GpuScene(ctx, sc)
        gs.frame()
        ctx.sync()
        ctx.capture_begin()
        gs.frame()
        g = ctx.capture_end()
        for _ in range(3):
            ctx.clear_colour(7)
            ctx.clear_depth(-0.5)
            ctx.sync()
            ctx.graph_launch(g, 1)
            ctx.sync()
            np.testing.assert_array_equal(ctx.read_colour(), f.colour)
            np.testing.assert_array_equal(ctx.read_depth().view(np.uint32), f.depth.view(np.uint32))
            gs.frame()
            ctx.sync()
