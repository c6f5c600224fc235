"""Shading waves of one draw and of several: draws of one programme, each with
its own uniforms and textures, lie over one another in a viewport whose edges
cut the shading blocks, alone and interleaved with another programme's.
Bit-exact against the oracle."""
import numpy as np
import pytest

import scenegen
from test_gpu_parity import assert_same

pytestmark = pytest.mark.gpu

N = pytest.importorskip("puresoft3d_amd.native")
from puresoft3d_amd import scenes as S  # noqa: E402

PROGS = [N.PROC_DEF01, N.PROC_DEF02, N.PROC_DEF03, N.PROC_DEF04, N.PROC_LAMBERT, N.PROC_BLINN, N.PROC_SHADOWED]


def draws_scene(prog, n_draws, seed, width, height, other=None):
    """n_draws meshes of random triangles, small and large; other: a programme
    whose draws come between"""
    sc = scenegen.micro_scene(prog, seed, width, height, n=6)
    sc.name = "draws_p%d_n%d_s%d_%dx%d_%s" % (prog, n_draws, seed, width, height, other)
    rng = np.random.default_rng(seed)
    lv = S.mip_levels(16, 16)
    sc.draws = []
    for k in range(n_draws):
        pos = scenegen.random_clip_triangles(rng, 30)
        u = {}
        if prog == N.PROC_DEF04:
            ang = rng.uniform(0, 2 * np.pi)
            R = np.eye(4)
            R[0, 0], R[0, 2], R[2, 0], R[2, 2] = np.cos(ang), np.sin(ang), -np.sin(ang), np.cos(ang)
            u[1] = S.colmajor(R)
        else:
            u[7] = S.vec4(*rng.uniform(-3, 3, 3), 0.0) if prog != N.PROC_LAMBERT else S.vec4(*rng.uniform(0.2, 0.9, 3))
            u[8] = S.vec4(*rng.uniform(-3, 3, 3), 0.0)
            u[9] = np.array([len(sc.textures)], np.int32)
            u[11] = np.array([int(rng.integers(1, 64))], np.int32)
            sc.textures.append(S.TextureSpec([S.noise_texture(16, seed + k, cells=4)], wrap=k & 1,
                                             levels=lv if k & 2 and prog in (N.PROC_BLINN, N.PROC_SHADOWED) else 1))
        sc.meshes["d%d" % k] = scenegen._slots_for(prog, pos, rng)
        sc.draws.append(S.DrawSpec("d%d" % k, prog, uniforms=u))
        if other is not None:
            sc.meshes["o%d" % k] = scenegen._slots_for(other, scenegen.random_clip_triangles(rng, 8), rng)
            sc.draws.append(S.DrawSpec("o%d" % k, other))
    return sc


@pytest.mark.parametrize("n_draws", [1, 2, 9])
@pytest.mark.parametrize("prog", PROGS)
def test_draws_of_a_programme(oracle, prog, n_draws):
    assert_same(draws_scene(prog, n_draws, 40 + prog, 47, 35), oracle)


@pytest.mark.parametrize("prog", [N.PROC_DEF03, N.PROC_BLINN, N.PROC_SHADOWED])
def test_draws_between_another_programmes(oracle, prog):
    assert_same(draws_scene(prog, 5, 60 + prog, 131, 18, other=N.PROC_DEF02), oracle)


def programmes_scene(seed, width, height, order):
    """small draws of the listed programmes, which share the waves that set
    their triangles up and those that shade them"""
    sc = scenegen.micro_scene(N.PROC_SHADOWED, seed, width, height, n=6)
    sc.name = "programmes_s%d_%dx%d_%s" % (seed, width, height, "_".join(map(str, order)))
    sky = scenegen.micro_scene(N.PROC_DEF04, seed + 1, width, height, n=6)
    sc.uniforms.update({0: sky.uniforms[0], 1: sky.uniforms[1], 2: np.array([len(sc.textures)], np.int32)})
    sc.textures += sky.textures
    rng = np.random.default_rng(seed)
    sc.draws = []
    for k, prog in enumerate(order):
        sc.meshes["p%d" % k] = scenegen._slots_for(prog, scenegen.random_clip_triangles(rng, 5 + 6 * (k % 4)), rng)
        u = {7: S.vec4(0.48, 0.6, 0.64)} if prog == N.PROC_LAMBERT else {}
        sc.draws.append(S.DrawSpec("p%d" % k, prog, uniforms=u))
    return sc


@pytest.mark.parametrize("order", [PROGS, PROGS[::-1] + PROGS * 2, [N.PROC_SHADOWED, N.PROC_DEF04], [N.PROC_LAMBERT, N.PROC_DEF03]])
def test_programmes_of_one_flush(oracle, order):
    assert_same(programmes_scene(80 + len(order), 131, 37, order), oracle)


def test_programmes_of_several_views():
    """views of one flush whose draws, of several programmes, share varyings:
    the images of the views rendered one by one"""
    w, h = 75, 37
    sc = programmes_scene(91, w, h, [N.PROC_BLINN, N.PROC_DEF04, N.PROC_DEF02, N.PROC_LAMBERT, N.PROC_BLINN])
    pv = [S.colmajor(np.diag([1.0 - 0.2 * k, 1.0, 1.0, 1.0])) for k in range(3)]
    ctx = N.Context(w, h)
    try:
        gs = S.GpuScene(ctx, sc)
        images = []
        for together in (False, True):
            views = [(ctx.texture_create(w, h, 4, wrap=N.CLAMP), ctx.texture_create(w, h, 4, wrap=N.CLAMP)) for _ in pv]
            for (c, d), m in zip(views, pv):
                ctx.target(c)
                ctx.depth_target(d)
                ctx.viewport(w, h)
                sc.uniforms[3] = m
                gs.frame(flush=not together)
            flushes = ctx.stats()["flushes"]
            ctx.flush()
            ctx.sync()
            assert not together or ctx.stats()["flushes"] == flushes + 1
            images.append([ctx.texture_download(t).ravel() for v in views for t in v])
    finally:
        ctx.close()
    assert any((a != images[0][0]).any() for a in images[0][2::2])   # the views differ
    for a, b in zip(*images):
        np.testing.assert_array_equal(a, b)
