"""The shading kernels' short forms of two steps against what they stand for:
1 / sqrt(x) with both operations rounded, and the clamped or wrapped texel pair
of a whole coordinate."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")


def selftest(op, a, b=None):
    ctx = N.Context(8, 8)
    try:
        return ctx.selftest_math(op, a, b) if b is not None else ctx.selftest_math(op, a)
    finally:
        ctx.close()


def test_reciprocal_root():
    """every float of the two binades that the range repeats, and floats of all
    magnitudes with the ends of the short form's range, zeros, infinity and NaN"""
    announce("selftest reciprocal root")
    rng = np.random.default_rng(5)
    two = np.arange(0x3f800000, 0x40800000, dtype=np.uint32)
    ends = np.array([0x0d800000, 0x71800000], np.uint32)   # 2^-100 and 2^100
    near = (ends[:, None].astype(np.int64) + np.arange(-64, 65)).ravel().astype(np.uint32)
    ones = (np.arange(256, dtype=np.uint32)[:, None] << 23 | np.array([0x7ffffd, 0x7ffffe, 0x7fffff, 0, 1], np.uint32)).ravel()
    x = np.concatenate([two, near, ones, rng.integers(0, 2**32, 1 << 20, dtype=np.uint64).astype(np.uint32),
                        np.array([0, 0x80000000, 1, 0x7f800000, 0xff800000, 0x7fc00000], np.uint32)]).view(np.float32)
    with np.errstate(all="ignore"):
        want = np.float32(1.0) / np.sqrt(x)
    got = selftest(11, x)
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


@pytest.mark.parametrize("wrap", [False, True])
def test_texel_pairs(wrap):
    """last texels 0 to 4095 and up to 2^22 - 1; coordinates around the multiples
    of the size, the float form's edge (+-2^21), the int32 extremes and beyond"""
    announce("selftest texel pairs wrap=%d" % wrap)
    rng = np.random.default_rng(7)
    ms, vs = [], []
    for m in list(range(0, 4096)) + [8191, 65534, 65535, (1 << 22) - 1]:
        q = rng.integers(-(1 << 21) // max(m, 1) - 2, (1 << 21) // max(m, 1) + 2, 6)
        v = np.concatenate([q * m, q * m - 1, q * m + 1, rng.integers(-(1 << 23), 1 << 23, 6), rng.integers(-2**31, 2**31, 6),
                            [0, -1, (1 << 21) - 1, 1 - (1 << 21), 1 << 21, -(1 << 21), 2**31 - 128, -2**31, 2**31, -2**33]])
        ms.append(np.full(v.size, m)); vs.append(v)
    m = np.concatenate(ms).astype(np.int64)
    x = np.concatenate(vs).astype(np.float32)
    x[::1009] = np.nan
    x[::1013] = -0.0
    with np.errstate(all="ignore"):
        v = np.where((x >= -2147483648.0) & (x < 2147483648.0), np.nan_to_num(x, posinf=0, neginf=0).astype(np.float64), -2147483648.0)
    v = v.astype(np.int64)
    v1 = ((v + 1 + 2**31) % 2**32) - 2**31
    if wrap:
        want = [np.where(m > 0, np.mod(k, np.maximum(m, 1)), 0) for k in (v, v1)]
    else:
        want = [np.clip(k, 0, m) for k in (v, v1)]
    b = (m.astype(np.uint32) | np.uint32(0x80000000 if wrap else 0)).view(np.float32)
    for op in (12, 13):
        got = selftest(op, x, b).view(np.int32)
        np.testing.assert_array_equal(got, want[op - 12].astype(np.int32))
