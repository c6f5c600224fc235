"""Clears without draws: up to eight fills come as kernel arguments, more from a
record buffer; and a sync with nothing logged after one that replayed."""
import numpy as np
import pytest

from conftest import announce
import scenegen

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


@pytest.mark.parametrize("n", [1, 8, 9])
def test_clears(n):
    announce("%d clears" % n)
    ctx = N.Context(64, 48)
    try:
        tex = [ctx.texture_create(33 + k, 17, 4, wrap=N.CLAMP) for k in range(n)]
        for k, t in enumerate(tex):
            ctx.target(t)
            ctx.clear_target(0x01020300 + k)
        ctx.target(N.DISPLAY)
        ctx.sync()
        ctx.sync()
        for k, t in enumerate(tex):
            got = ctx.texture_download(t).view(np.uint32)
            assert (got == 0x01020300 + k).all()
    finally:
        ctx.close()


def test_statistics_after_replays(oracle):
    """a flush that overflows its scratch is replayed and counted once, and so is the next one"""
    sc = scenegen.micro_scene(N.PROC_BLINN, 5)
    announce("replay " + sc.name)
    _, want = oracle.render_scene(sc)
    ctx = N.Context(sc.width, sc.height, flags=1)   # PSGPU_CREATE_TINY_SCRATCH
    try:
        gs = S.GpuScene(ctx, sc)
        for frame in range(3):
            ctx.reset_stats()
            gs.frame()
            f = ctx.fence()
            ctx.fence_wait(f)
            ctx.sync()
            st = ctx.stats()
            assert st["frags_shaded"] == want.frags_shaded and st["tris_culled"] == want.tris_culled
            assert (st["retries"] > 0) == (frame == 0)
    finally:
        ctx.close()
