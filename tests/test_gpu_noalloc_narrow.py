"""psgpu_sync_noalloc on many narrow views in one flush: nothing that only
widens accesses may take scratch from what fits into the fixed array.  The
views' colours and depths against psgpu_sync's, bit for bit."""
import numpy as np
import pytest

from conftest import announce
import scenegen

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


def _render(sizes, noalloc):
    # six triangles across every view, of some hundred rows where a view is very tall
    rng = np.random.default_rng(5)
    sc = scenegen.micro_scene(N.PROC_DEF02, 5, 64, 64, n=24)
    pos = np.zeros((6, 3, 4), np.float32)
    pos[..., 0] = rng.uniform(-1, 1, (6, 3)) + [-20.0, 20.0, 0.0]
    pos[..., 1] = rng.uniform(-0.9, 0.9, (6, 1)) + rng.uniform(-1, 1, (6, 3)) * (0.0002 if sizes[0][1] > 1000 else 1.0)
    pos[..., 2] = rng.uniform(-0.9, 0.9, (6, 1))
    pos[..., 3] = 1.0
    sc.meshes["m"] = scenegen._slots_for(N.PROC_DEF02, pos.reshape(-1, 4), rng)
    sc.uniforms[4] = S.colmajor(np.eye(4))
    sc.draws = sc.draws[:1]
    sc.draws[0].behavior = N.UPDATE_DEPTH | N.TEST_DEPTH
    with N.Context(64, 64) as ctx:
        gs = S.GpuScene(ctx, sc)
        targets = [(w, h, ctx.texture_create(w, h, 4, wrap=N.CLAMP), ctx.texture_create(w, h, 4, wrap=N.CLAMP))
                   for w, h in sizes]
        ctx.sync()
        for w, h, colour, depth in targets:
            ctx.target(colour)
            ctx.depth_target(depth)
            ctx.viewport(w, h)
            ctx.clear_depth(1.0)
            ctx.clear_target(0x00302010)
            gs.frame(clear=False, flush=False)
        if noalloc:
            ctx.sync_noalloc()
        else:
            ctx.sync()
        return [(ctx.texture_download(c), ctx.texture_download(d)) for _, _, c, d in targets], ctx.stats()


# nine planes of 2 x 10^6 pixels are 72 MB, and 288 MB with rows of eight
@pytest.mark.parametrize("sizes", [[(2, 1000000)] * 9, [(3, 50), (31, 37), (4, 9), (66, 21), (2, 200)]])
def test_narrow_views(sizes):
    announce("sync_noalloc %d views, first %dx%d" % (len(sizes), sizes[0][0], sizes[0][1]))
    got, st = _render(sizes, True)
    want, ost = _render(sizes, False)
    for (gc, gd), (wc, wd) in zip(got, want):
        np.testing.assert_array_equal(gc, wc)
        np.testing.assert_array_equal(gd, wd)
    assert st["frags_shaded"] == ost["frags_shaded"] > 0
    assert st["frags_rasterised"] == ost["frags_rasterised"]
