"""Span and piece kernels on wide spans: triangles many tiles wide beside tiny
ones, spans at the length where varying checkpoints begin, every number of
varyings, and tiles that hundreds of one-span runs share.  Bit-exact against
the oracle."""
import numpy as np
import pytest

import scenegen
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")


def wide_scene(prog, n, width, height, seed, lengths=False):
    """n triangles that reach far off screen, n / 2 tiny ones between them;
    lengths: triangles 40 to 60 pixels wide instead"""
    sc = scenegen.micro_scene(prog, seed, width, height, n=24)
    sc.name = "wide_p%d_%d_%dx%d_s%d_%d" % (prog, n, width, height, seed, lengths)
    rng = np.random.default_rng(seed)
    if lengths:
        big = np.zeros((n, 3, 4), np.float32)
        for t in range(n):
            x0, w = rng.uniform(-1, 0.9), rng.uniform(40, 60) * 2 / width
            big[t, :, 0] = x0, x0 + w, x0 + w * rng.uniform(0, 1)
            big[t, :, 1] = rng.uniform(-1, 1, 3)
            big[t, :, 2] = rng.uniform(-0.5, 0.5)
        big[:, :, 3] = 1.0
    else:
        big = scenegen.random_clip_triangles(rng, n, kind=4).reshape(n, 3, 4)
    pos = np.concatenate([big, scenegen.random_clip_triangles(rng, n // 2, kind=1).reshape(-1, 3, 4)], 0)
    pos = pos[rng.permutation(len(pos))].reshape(-1, 4)
    sc.meshes["m"] = scenegen._slots_for(prog, pos, rng)
    sc.draws = sc.draws[:1]
    sc.draws[0].behavior = N.UPDATE_DEPTH | N.TEST_DEPTH
    return sc


@pytest.mark.parametrize("prog", [N.PROC_DEF03, N.PROC_DEF05, N.PROC_LAMBERT, N.PROC_BLINN, N.PROC_CLOUD,
                                  N.PROC_CLOUD_SHADOW])
@pytest.mark.parametrize("lengths", [False, True])
def test_wide_spans(oracle, prog, lengths):
    assert_same(wide_scene(prog, 40, 1507, 37, 3 + prog, lengths), oracle)


@pytest.mark.parametrize("tiling", [(1, 8, 2), (2, 16, 1), (8, 8, 1), (16, 2, 2), (64, 1, 1)])
def test_wide_span_tilings(oracle, tiling):
    assert_same(wide_scene(N.PROC_BLINN, 30, 1102, 70, 9), oracle, tiling=tiling)


# four to five of eight rows a triangle: 64, 256 and more runs a tile
@pytest.mark.parametrize("n", [14, 60, 500])
def test_wide_span_runs(oracle, n):
    assert_same(wide_scene(N.PROC_DEF02, n, 200, 8, n), oracle)
