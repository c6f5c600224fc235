"""Raster kernel on crowded tiles: a viewport of one to a few tiles that
hundreds of overlapping triangles share, so that a tile's runs are taken from
the lanes (up to 64), sorted in LDS (up to 256) and sorted in memory (beyond),
its pieces overlap within a batch, and draws with and without depth test and
update alternate.  Bit-exact against the oracle."""
import numpy as np
import pytest

from conftest import announce
import scenegen
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


def crowded_scene(n, width, height, seed, mixed):
    """n triangles a draw, a third of them tiny; mixed: four draws, one of
    each combination of depth test and update"""
    sc = scenegen.micro_scene(N.PROC_DEF02, seed, width, height, n=24)
    sc.name = "crowded_%d_%dx%d_s%d_%d" % (n, width, height, seed, mixed)
    rng = np.random.default_rng(seed)
    pos = np.concatenate([scenegen.random_clip_triangles(rng, n - n // 3, kind=0),
                          scenegen.random_clip_triangles(rng, n // 3, kind=1)], 0).reshape(-1, 3, 4)
    pos = pos[rng.permutation(n)].reshape(-1, 4)
    sc.meshes["m"] = scenegen._slots_for(N.PROC_DEF02, pos, rng)
    full = N.UPDATE_DEPTH | N.TEST_DEPTH
    order = [full, N.TEST_DEPTH, N.UPDATE_DEPTH, full] if mixed else [full]
    sc.draws = [S.DrawSpec("m", N.PROC_DEF02, behavior=b) for b in order]
    return sc


# rows of a triangle here: about 5 of 8, so 64 row items are some 13 triangles
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [40, 700, 820, 840, 3000, 5000])
def test_crowded_tile(oracle, n, mixed):
    assert_same(crowded_scene(n, 31, 8, n, mixed), oracle)


@pytest.mark.parametrize("tiling", [(1, 8, 8), (2, 16, 1), (8, 8, 8), (8, 64, 3), (16, 4, 5), (32, 2, 3), (64, 1, 1)])
def test_crowded_tilings(oracle, tiling):
    announce("crowded %s" % (tiling,))
    assert_same(crowded_scene(1500, 47, 35, 5, True), oracle, tiling=tiling)
