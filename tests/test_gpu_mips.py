"""Mip chains at the edges of the kernel's 64 x 64 squares and of its six levels
a launch: sides of one texel, odd sides, long thin textures, both texel sizes,
several layers.  Against the definition, byte for byte."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402


def next_level(a):
    """rounded mean of 2 x 2 texels; a side halves rounding down, to at least 1"""
    h, w = a.shape[:2]
    y, x = np.arange(max(1, h // 2)) * 2, np.arange(max(1, w // 2)) * 2
    y1, x1 = np.minimum(y + 1, h - 1), np.minimum(x + 1, w - 1)
    v = a.astype(np.int32)
    s = v[y][:, x] + v[y][:, x1] + v[y1][:, x] + v[y1][:, x1]
    return ((s + 2) >> 2).astype(np.uint8)


@pytest.mark.parametrize("elem", [4, 1])
@pytest.mark.parametrize("w,h,layers", [(1, 2, 1), (1, 700, 2), (333, 1, 1), (2, 64, 1), (63, 65, 3), (64, 64, 6),
                                        (65, 129, 1), (127, 190, 1), (128, 3, 2), (4100, 5, 1), (260, 4097, 1)])
def test_mip_chain(w, h, layers, elem):
    announce("mips %dx%d x%d, %d bytes" % (w, h, layers, elem))
    rng = np.random.default_rng(w * 5 + h)
    lv = S.mip_levels(w, h)
    ctx = N.Context(8, 8)
    try:
        t = ctx.texture_create(w, h, elem, extra_layers=layers - 1, mip_levels=lv)
        want = [rng.integers(0, 256, (h, w, elem), dtype=np.uint8) for _ in range(layers)]
        for k in range(layers):
            ctx.texture_upload(t, want[k], layer=k)
        ctx.texture_generate_mips(t)
        for k in range(layers):
            a = want[k]
            for level in range(lv):
                got = ctx.texture_download(t, layer=k, level=level)
                np.testing.assert_array_equal(got.reshape(a.shape), a, err_msg="layer %d level %d" % (k, level))
                a = next_level(a)
    finally:
        ctx.close()
