"""Recorded command lists with more commands than the log has flag words
(16,384): the eager run of the recording and the one after a change of tiling
end the log in between, with work logged before the recording in it as well.
Pixels and statistics as of the same commands without a recording."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402

FLAG_WORDS = 16384


@pytest.mark.parametrize("before", [0, 7])
def test_recording_longer_than_the_log(oracle, before):
    sc = S.sphere_scene(width=64, height=48, tex_size=16)
    announce("recording of %d commands after %d" % (FLAG_WORDS + 4, before))
    want, _ = oracle.render_scene(sc)
    with N.Context(sc.width, sc.height) as ctx:
        gs = S.GpuScene(ctx, sc)
        ctx.sync()
        for k in range(before):
            ctx.clear_colour(k)
            ctx.flush()
        ctx.reset_stats()
        ctx.capture_begin()
        gs.frame()
        first = ctx.stats()["tris_in"]
        for k in range(FLAG_WORDS + 2):      # one command each
            ctx.clear_colour(0x01000000 + k)
            ctx.flush()
        gs.frame()
        graph = ctx.capture_end()
        np.testing.assert_array_equal(ctx.read_colour(), want.colour)
        shaded = ctx.stats()["frags_shaded"]
        assert first > 0 and shaded > 0 and shaded % 2 == 0
        for k in range(2):                   # replayed, then run eagerly once more
            if k:
                ctx.tiling(8, 8, 1)
            ctx.clear_colour(5)
            ctx.graph_launch(graph)
            np.testing.assert_array_equal(ctx.read_colour(), want.colour)
            np.testing.assert_array_equal(ctx.read_depth().view(np.uint32), want.depth.view(np.uint32))
            assert ctx.stats()["frags_shaded"] == (k + 2) * shaded
        ctx.graph_destroy(graph)
