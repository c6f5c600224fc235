"""What a program that uses this package has it do, as cases that can be timed.

A case is a dict of plain values.  Five kinds of work are covered, each
through the calls a program makes:

  frame   one view drawn into the display: clear, the scene's draws, flush.
          Either call by call with a wait at the end of the frame (what the
          reference's synchronous drawVAO programs do), or recorded once and
          replayed as a graph (a program that redraws a static draw list)
  views   many views of resident scenes in one graph launch, each into its
          own colour and depth textures
  serve   a burst of view requests through the serving loop, images delivered
          to host memory
  shade   one step of the differentiable shading: forward, L2 loss, backward
  mips    the mip chain of a texture whose level 0 changed

prepare() makes inputs from the seed alone; run() is one pass.  A frame's
outputs are the display and the depth buffer where they lie in device memory.
"""
import ctypes
import math

import numpy as np
import torch

from puresoft3d_amd import adjoint as A
from puresoft3d_amd import native as N
from puresoft3d_amd import scenes as S
from puresoft3d_amd import serving as SV


def _frame(name, scene, width, height, cells, objects, tex, graph, chunk=0, rows=0, waves=0):
    """chunk, rows, waves: the raster tiling, 0 for the library's default"""
    return {"name": name, "kind": "frame", "scene": scene, "width": width, "height": height, "cells": cells,
            "objects": objects, "tex": tex, "graph": graph, "chunk": chunk, "rows": rows, "waves": waves}


def listed():
    return [
        # the smallest call: one textured sphere of 2,048 triangles, drawn call by call and waited for
        _frame("sphere_640x480", "sphere", 640, 480, 32, 1, 512, False),
        # the plain path of a viewer: one small view of odd size, drawn call by call and waited for
        _frame("view_515x389", "terrain", 515, 389, 140, 6, 1024, False),
        # the benchmark's frame: 200k triangles, 2048^2 mipmapped maps, recorded, in the tiling its tuner picks
        _frame("terrain_1920x1080", "terrain", 1920, 1080, 300, 64, 2048, True, 2, 16, 1),
        # the largest frame: 4K, half a million triangles, the library's default tiling
        _frame("terrain_3840x2160", "terrain", 3840, 2160, 490, 64, 2048, True),
        # two passes: a 512^2 shadow map, then the scene lit through it
        _frame("shadow_1280x720", "shadow", 1280, 720, 200, 24, 1024, True),
        # a blended layer over a shadowed scene, its shadow pass discarding (the demo's cloud)
        _frame("cloud_960x540", "cloud", 960, 540, 120, 12, 512, True),
        # the reference's own programmes in one frame: textured, coloured and bump-mapped objects before a skybox
        _frame("demo_1366x768", "demo", 1366, 768, 48, 24, 512, True),
        # many views of resident scenes in one launch, areas 256^2 to 1024^2, 10k to 300k triangles each
        {"name": "views_32", "kind": "views", "views": 32, "scenes": 8, "side_lo": 256, "side_hi": 1024,
         "tri_lo": 10000, "tri_hi": 300000, "tex": 1024},
        # a burst of requests served to host memory, areas 128^2 to 1024^2, 1k to 200k triangles each
        {"name": "serve_48", "kind": "serve", "views": 48, "scenes": 8, "side_lo": 128, "side_hi": 1024,
         "tri_lo": 1000, "tri_hi": 200000, "tex": 1024},
        # learning a texture and two material parameters: 512^2 image, 1024^2 texture
        {"name": "shade_512", "kind": "shade", "width": 512, "height": 512, "tex_w": 1024, "tex_h": 1024},
        # the same close up and odd: many pixels of a larger image on each texel of a small texture
        {"name": "shade_1237x891", "kind": "shade", "width": 1237, "height": 891, "tex_w": 250, "tex_h": 130},
        # the mip chains of a cube map whose faces were drawn anew
        {"name": "mips_1024x6", "kind": "mips", "width": 1024, "height": 1024, "layers": 6},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi):
    """a width and height with the area log-uniform in [lo^2, hi^2]; the
    display refuses widths of 4k + 1 (its default depth row would be shorter
    than the row)"""
    area = _log(rng, lo * lo, hi * hi)
    asp = _log(rng, 0.75, 2.4)
    w = max(16, int(round(math.sqrt(area * asp))))
    h = max(16, int(round(area / w)))
    return (w + 1 if w % 4 == 1 else w), h


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "views", "serve", "shade", "shade", "mips"])
    if kind == "frame":
        scene = rng.choice(["sphere", "terrain", "terrain", "shadow", "cloud", "demo"])
        w, h = _size(rng, 128, 1600 if scene in ("sphere", "terrain") else 900)
        cells = int(round({"sphere": _log(rng, 8, 100), "terrain": _log(rng, 12, 400), "shadow": _log(rng, 12, 250),
                           "cloud": _log(rng, 12, 150), "demo": _log(rng, 8, 64)}[scene]))
        chunk, rows, waves = rng.choice([(0, 0, 0), (0, 0, 0), (2, 16, 1), (2, 8, 2), (4, 16, 2), (8, 8, 1)])
        return dict(_frame("", scene, w, h, cells, rng.randint(1, 24), rng.choice([128, 256, 512, 1024]),
                           rng.random() < 0.6, chunk, rows, waves))
    if kind in ("views", "serve"):
        lo = int(_log(rng, 64, 256))
        return {"name": "", "kind": kind, "views": rng.randint(3, 28), "scenes": rng.randint(1, 8), "side_lo": lo,
                "side_hi": min(1024, lo * rng.choice([1, 2, 4])), "tri_lo": 1000,
                "tri_hi": int(_log(rng, 2000, 200000)), "tex": rng.choice([256, 512, 1024])}
    if kind == "shade":
        w, h = _size(rng, 40, 1300)
        return {"name": "", "kind": "shade", "width": w - rng.randint(0, 1), "height": h,
                "tex_w": int(_log(rng, 4, 2048)), "tex_h": int(_log(rng, 4, 2048))}
    return {"name": "", "kind": "mips", "width": int(_log(rng, 2, 2048)), "height": int(_log(rng, 2, 2048)),
            "layers": rng.randint(1, 6)}


# ---------------------------------------------------------------- inputs
def _maps(tex, seed, repeat=True):
    """albedo and normal map of side tex with full mip chains: a seeded
    periodic tile repeated, so that the memory footprint is the full size"""
    lv = S.mip_levels(tex, tex)
    return [S.TextureSpec([S.tiled_texture(lambda t, s: S.noise_texture(t, s, cells=16, octaves=3), tex, seed, 256)],
                          wrap=N.WRAP, levels=lv),
            S.TextureSpec([S.tiled_texture(lambda t, s: S.normal_map(t, s, cells=16), tex, seed + 1, 256)],
                          wrap=N.WRAP, levels=lv)]


def _demo_scene(case, seed):
    """objects of the reference's textured, per-vertex-coloured and
    bump-mapped programmes, interleaved, in front of a skybox"""
    rng = np.random.default_rng(seed)
    w, h, n = case["width"], case["height"], case["cells"]
    sc = S.Scene(w, h)
    m = S.uv_sphere(n, n, 1.0, tangents=True)
    sc.meshes["tex"] = {0: m[0], 3: m[3], 4: m[4]}
    sc.meshes["col"] = {0: m[0], 1: m[3], 2: rng.uniform(0, 255, (m[0].shape[0], 4)).astype(np.float32)}
    sc.meshes["bump"] = m
    sc.meshes["sky"] = {0: np.array([[-1, -1, 0.999, 1], [1, -1, 0.999, 1], [1, 1, 0.999, 1],
                                     [-1, -1, 0.999, 1], [1, 1, 0.999, 1], [-1, 1, 0.999, 1]], np.float32)}
    t = case["tex"]
    sc.textures.append(S.TextureSpec([S.tiled_texture(S.noise_texture, t, seed, 256)], wrap=N.WRAP))
    sc.textures.append(S.TextureSpec([S.tiled_texture(S.normal_map, t, seed + 1, 256)], wrap=N.WRAP))
    sc.textures.append(S.TextureSpec([S.tiled_texture(S.noise_texture, t, seed + 2 + k, 128) for k in range(6)],
                                     wrap=N.CLAMP))
    eye = (0.4, 1.3, 9.0)
    sc.uniforms[1] = S.colmajor(S.look_at((0, 0, 0), (0.6, 0.3, -1.0)))
    sc.uniforms[2] = np.array([2], np.int32)
    sc.uniforms[3] = S.colmajor(S.perspective(np.radians(60.0), w / h, 0.1, 50.0) @ S.look_at(eye, (0, 0, 0)))
    sc.uniforms[7] = S.vec4(6.0, 8.0, 10.0, 0.0)
    sc.uniforms[8] = S.vec4(*eye, 0.0)
    sc.uniforms[9] = np.array([0], np.int32)
    sc.uniforms[10] = np.array([1], np.int32)
    progs = [("tex", N.PROC_DEF01), ("col", N.PROC_DEF02), ("bump", N.PROC_DEF03)]
    for k in range(case["objects"]):
        a = rng.uniform(0, 2 * np.pi)
        R = np.eye(4)
        R[0, 0], R[0, 2], R[2, 0], R[2, 2] = np.cos(a), np.sin(a), -np.sin(a), np.cos(a)
        mesh, prog = progs[k % 3]
        at = S.translate(rng.uniform(-6, 6), rng.uniform(-3, 3), rng.uniform(-6, 3))
        sc.draws.append(S.DrawSpec(mesh, prog, {4: S.colmajor(at @ R), 5: S.colmajor(R)}))
    sc.draws.append(S.DrawSpec("sky", N.PROC_DEF04))
    return sc


def _shadow_side(case):
    """the shadow map: a power of two that the display covers (the pass leaves the colour target bound)"""
    return min(case["tex"], 1 << (min(case["width"], case["height"]).bit_length() - 1))


def _scene(case, seed):
    w, h, cells, n, tex = (case[k] for k in ("width", "height", "cells", "objects", "tex"))
    smap = _shadow_side(case)
    if case["scene"] == "sphere":
        sc = S.sphere_scene(w, h, seed, 16)
        sc.meshes["sphere"] = S.uv_sphere(cells, cells, 1.0, seed=seed)
        sc.textures[0] = S.TextureSpec([S.tiled_texture(S.noise_texture, tex, seed, 256)], wrap=N.WRAP)
        return sc
    if case["scene"] == "demo":
        return _demo_scene(case, seed)
    if case["scene"] == "terrain":
        sc = S.terrain_scene(w, h, seed, cells, n, 16)
    elif case["scene"] == "shadow":
        sc = S.shadow_terrain_scene(w, h, seed, cells, n, 16, smap)
    else:
        sc = S.cloud_terrain_scene(w, h, seed, cells, n, 16, smap, cloud_cells=max(2, cells // 4),
                                   cloud_tex=min(tex, 256))
    sc.textures[:2] = _maps(tex, seed + 1)
    return sc


def _assets(case, seed):
    """resident terrain patches; their triangle counts, log-uniform in [tri_lo, tri_hi], are the case's"""
    rng = np.random.default_rng(11)
    out = []
    for k in range(case["scenes"]):
        T = math.exp(rng.uniform(math.log(case["tri_lo"]), math.log(case["tri_hi"])))
        cells = max(2, int(round(math.sqrt(T / 2.0))))
        mesh = S.terrain(cells, 40.0, seed * 100 + k, height=4.0, uv_repeat=4.0)[0]
        out.append(S.SceneAsset(mesh, _maps(case["tex"], seed * 100 + 2 * k), np.zeros(3), 28.0, "patch%d" % k))
    return out


def _views(case, seed, assets):
    """scenes and cameras from the seed, sizes from the case"""
    sizes = S.batch_views(assets, case["views"], 12, case["side_lo"], case["side_hi"])
    views = S.batch_views(assets, case["views"], seed + 1, case["side_lo"], case["side_hi"])
    for v, z in zip(views, sizes):
        v.width, v.height = z.width, z.height
    return views


class _Device:
    """device memory that `owner` holds, in the form torch reads; keeps the owner alive"""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, ptr, shape, typestr):
    return torch.as_tensor(_Device(owner, ptr, shape, typestr), device="cuda")


def _display(ctx):
    """the display (BGRA8, rows top-down) and the default depth buffer"""
    p, scan = ctypes.c_void_p(), ctypes.c_int()
    ctx.L.psgpu_display_device_ptr(ctx.h, ctypes.byref(p))
    colour = _tensor(ctx, p.value, (ctx.height, ctx.width, 4), "|u1")
    ctx.L.psgpu_depth_device_ptr(ctx.h, ctypes.byref(p), ctypes.byref(scan))
    return colour, _tensor(ctx, p.value, (ctx.height, scan.value), "<f4")


def _target_ptrs(ctx, colour, depth, w, h):
    """device addresses of a pair of target textures, as a post-processor sees them"""
    seen = []

    def see(frame, stream):
        seen.append((frame.colour, frame.depth))
        return 0
    ctx.target(colour)
    ctx.depth_target(depth)
    ctx.viewport(w, h)
    ctx.post_process(see)
    ctx.target(N.DISPLAY)
    ctx.depth_target(N.DEFAULT_DEPTH)
    ctx.viewport(ctx.width, ctx.height)
    ctx.sync()
    return seen[0]


def _shade_inputs(case, seed):
    """Texture, parameters, target image and geometry buffer of the learning
    step.  The geometry buffer is that of a unit sphere, ray cast in 64 bits:
    per pixel normal, 1 | world position, 0 | texture coordinates, 0, 0, rows
    bottom-up; zero where the ray misses."""
    w, h = case["width"], case["height"]
    rng = np.random.default_rng(seed)
    eye = np.array([0.3 * rng.uniform(-1, 1), 0.4, 3.0])
    view = S.look_at(eye, (0.0, 0.0, 0.0))[:3, :3]
    f = math.tan(math.radians(45.0) / 2.0)
    x, y = np.meshgrid((np.arange(w) + 0.5) / w * 2 - 1, (np.arange(h) + 0.5) / h * 2 - 1)
    d = np.stack([x * f * w / h, y * f, -np.ones_like(x)], -1) @ view
    d /= np.linalg.norm(d, axis=-1, keepdims=True)
    b = d @ eye
    disc = b * b - (eye @ eye - 1.0)
    hit = disc > 0
    p = eye + (-b - np.sqrt(np.where(hit, disc, 0.0)))[..., None] * d
    g = np.zeros((h, w, 12))
    g[..., 0:3], g[..., 3], g[..., 4:7] = p, 1.0, p
    g[..., 8] = np.arctan2(p[..., 2], p[..., 0]) / (2 * np.pi) % 1.0
    g[..., 9] = np.arccos(np.clip(p[..., 1], -1, 1)) / np.pi
    g[~hit] = 0.0
    tex = 0.25 + 0.5 * rng.random((case["tex_h"], case["tex_w"], 3))
    target = np.where(hit[..., None], 0.2 + 0.6 * rng.random((h, w, 3)), 0.0)
    return {"gbuf": g.astype(np.float32), "tex": tex.astype(np.float32), "target": target.astype(np.float32),
            "params": np.array([1.0, 12.0], np.float32), "eye": eye, "light": np.array([4.0, 5.0, 6.0]), "ks": 0.5}


class _Server(SV.RenderServer):
    """gives its pooled targets back before its context goes"""

    def __del__(self):
        self.close()


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        sc = _scene(case, seed)
        ctx = N.Context(sc.width, sc.height)
        if case["chunk"]:
            ctx.tiling(case["chunk"], case["rows"], case["waves"])
        gs = S.GpuScene(ctx, sc)
        graph = None
        if case["graph"]:
            ctx.capture_begin()
            gs.frame(flush=False)
            graph = ctx.capture_end()
        return {"kind": kind, "ctx": ctx, "scene": gs, "graph": graph, "out": _display(ctx)}
    if kind == "views":
        ctx = N.Context(64, 64)
        assets = _assets(case, seed)
        views = _views(case, seed, assets)
        b = S.GpuBatch(ctx, assets, views)
        ctx.capture_begin()
        b.submit()
        graph = ctx.capture_end()
        out = []
        for v, (c, d) in zip(views, b.targets):
            pc, pd = _target_ptrs(ctx, c, d, v.width, v.height)
            out.append((_tensor(ctx, pc, (v.height, v.width, 4), "|u1"), _tensor(ctx, pd, (v.height, v.width), "<f4")))
        return {"kind": kind, "ctx": ctx, "batch": b, "graph": graph, "out": out}
    if kind == "serve":
        ctx = N.Context(64, 64)
        assets = _assets(case, seed)
        views = _views(case, seed, assets)
        srv = _Server(ctx, assets)
        srv.serve(views, np.zeros(len(views)))     # the server's pools, as in a server that has been running
        return {"kind": kind, "ctx": ctx, "server": srv, "views": views, "arrivals": np.zeros(len(views))}
    if kind == "shade":
        i = _shade_inputs(case, seed)
        ctx = N.Context(64, 64)
        gb = A.GeometryBuffer(ctx, S.uv_sphere(8, 8, 1.0, tangents=True), case["width"], case["height"], i["eye"],
                              light=i["light"])
        gb.gbuf.copy_(torch.from_numpy(i["gbuf"]))
        dev = {k: torch.from_numpy(i[k]).cuda() for k in ("tex", "params", "target")}
        return {"kind": kind, "ctx": ctx, "gb": gb, "ks": i["ks"], "target": dev["target"],
                "tex": dev["tex"].requires_grad_(), "params": dev["params"].requires_grad_()}
    w, h, layers = case["width"], case["height"], case["layers"]
    rng = np.random.default_rng(seed)
    ctx = N.Context(64, 64)
    lv = S.mip_levels(w, h)
    tex = ctx.texture_create(w, h, 4, extra_layers=layers - 1, wrap=N.WRAP, mip_levels=lv)
    for k in range(layers):
        ctx.texture_upload(tex, rng.integers(0, 256, (h, w, 4), dtype=np.uint8), layer=k)
    # the texture's memory: each layer its levels one after the other, padded to 256 bytes
    size = sum(max(1, w >> l) * max(1, h >> l) * 4 for l in range(lv))
    depth = ctx.texture_create(w, h, 4)
    ptr, _ = _target_ptrs(ctx, tex, depth, w, h)
    return {"kind": kind, "ctx": ctx, "tex": tex, "out": _tensor(ctx, ptr, (layers, (size + 255) // 256 * 256), "|u1")}


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "frame":
        if state["graph"] is not None:
            ctx.graph_launch(state["graph"])
        else:
            state["scene"].frame()
            ctx.sync()
        return {"colour": state["out"][0], "depth": state["out"][1]}
    if kind == "views":
        ctx.graph_launch(state["graph"])
        return state["out"]
    if kind == "serve":
        _, _, images = state["server"].serve(state["views"], state["arrivals"], keep=range(len(state["views"])))
        return [images[k] for k in range(len(images))]
    if kind == "shade":
        image = A.shade(state["tex"], state["params"], state["gb"], state["ks"])
        loss = ((image - state["target"]) ** 2).sum()
        gtex, gparams = torch.autograd.grad(loss, [state["tex"], state["params"]])
        return {"image": image.detach(), "loss": loss.detach(), "grad_tex": gtex, "grad_params": gparams}
    ctx.texture_generate_mips(state["tex"])
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without
_VERTEX = {"sphere": 40, "terrain": 72, "shadow": 72, "cloud": 72, "demo": 56}   # bytes a vertex, on average


def work(case):
    """bytes: vertex streams, texels that the pixels can touch, colour and
    depth, each once; flops: some 600 a triangle (transform, set-up) and some
    250 a pixel (interpolation, filtering, lighting)"""
    kind = case["kind"]
    if kind == "shade":
        px, tx = case["width"] * case["height"], case["tex_w"] * case["tex_h"]
        # forward and backward each read the geometry; image, target, its gradient; texture and its gradient
        return {"bytes": px * (48 + 12 * 2) + tx * 12 * 2, "flops": px * 300}
    if kind == "mips":
        px = case["width"] * case["height"] * case["layers"]
        return {"bytes": px * 4 * 4 // 3 + px * 4 // 3, "flops": px * 4 * 2}
    if kind == "frame":
        px = case["width"] * case["height"]
        c, n = case["cells"], case["objects"]
        tris = {"sphere": 2 * c * c, "demo": n * 2 * c * c}.get(case["scene"], 2 * c * c + 320 * n)
        maps = 4 * case["tex"] ** 2 * (8 if case["scene"] == "demo" else 1 if case["scene"] == "sphere" else 2)
        vertex, passes = _VERTEX[case["scene"]], 2 if case["scene"] in ("shadow", "cloud") else 1
        out = px * 8 + (_shadow_side(case) ** 2 * 4 if passes == 2 else 0)
        return {"bytes": tris * 3 * vertex * passes + min(maps * 4 // 3, 64 * px) + out,
                "flops": tris * 600 * passes + px * 250}
    mean = lambda lo, hi: (hi - lo) / math.log(hi / lo) if hi > lo else lo  # noqa: E731  of a log-uniform value
    px = case["views"] * mean(case["side_lo"] ** 2, case["side_hi"] ** 2)
    tris = case["views"] * mean(case["tri_lo"], case["tri_hi"])
    # a scene's streams and maps are read once, however many views show it
    streams = case["scenes"] * mean(case["tri_lo"], case["tri_hi"]) * 3 * 72
    return {"bytes": streams + min(case["scenes"] * 2 * case["tex"] ** 2 * 4 * 4 // 3, 64 * px) + px * 8,
            "flops": tris * 600 + px * 250}


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    """The shading step in 64 bits.  The other kinds answer with colour bytes,
    which are whole numbers, and with depths whose value at a pixel hangs on
    which fragments the FP32 coverage and depth rules let through: they have
    no 64-bit counterpart."""
    if case["kind"] != "shade":
        return None
    i = _shade_inputs(case, seed)
    c = lambda v: torch.from_numpy(np.asarray(v)).cuda().double()  # noqa: E731
    g, target = c(i["gbuf"]), c(i["target"])
    tex, params = c(i["tex"]).requires_grad_(), c(i["params"]).requires_grad_()
    norm = lambda v: v / v.norm(dim=-1, keepdim=True)  # noqa: E731
    hit = g[..., 3] != 0
    n, p, uv = norm(g[hit][:, 0:3]), g[hit][:, 4:7], g[hit][:, 8:10]
    # the program hands light and camera over as 32-bit numbers
    L, E = (norm(c(i[k].astype(np.float32)) - p) for k in ("light", "eye"))
    H = norm(L + E)
    lam, s = (n * L).sum(-1).clamp(min=0), (n * H).sum(-1).clamp(min=0)
    h, w = tex.shape[:2]
    x, y = uv[:, 0] * w, uv[:, 1] * h
    x0, y0 = x.floor(), y.floor()
    ax, ay = (x - x0)[:, None], (y - y0)[:, None]
    c0, r0 = x0.long() % w, y0.long() % h
    c1, r1 = (c0 + 1) % w, (r0 + 1) % h
    t = ((tex[r0, c0] * (1 - ax) + tex[r0, c1] * ax) * (1 - ay) + (tex[r1, c0] * (1 - ax) + tex[r1, c1] * ax) * ay)
    spec = torch.where(s > 0, i["ks"] * s.clamp(min=1e-300) ** params[1], torch.zeros_like(s))
    image = torch.zeros(g.shape[:2] + (3,), dtype=torch.float64, device="cuda")
    image = image.masked_scatter(hit[..., None], params[0] * t * lam[:, None] + spec[:, None])
    loss = ((image - target) ** 2).sum()
    gtex, gparams = torch.autograd.grad(loss, [tex, params])
    return {"image": image.detach(), "loss": loss.detach(), "grad_tex": gtex, "grad_params": gparams}
