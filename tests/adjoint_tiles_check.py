"""Backward pass of the adjoint over image and texture sizes at the edges of
its tiles, run in a process of its own by tests/test_adjoint_tiles.py (torch
must be imported before libpsgpu loads).  Prints one JSON line per case: the
relative errors of the texel and parameter gradients against the FP64 oracle."""
import json
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))

from puresoft3d_amd import adjoint as A  # noqa: E402
from puresoft3d_amd import native as N  # noqa: E402
from puresoft3d_amd import scenes as S  # noqa: E402
import pyoracle  # noqa: E402

# image, texture, texels a pixel, how the texture coordinates run over it
CASES = [
    (1, 1, 1, 1, 1.0, "smooth"),
    (32, 32, 7, 5, 0.2, "smooth"),
    (33, 31, 49, 67, 1.1, "seam"),         # 50 x 68 texels: the largest texture kept in LDS
    (65, 64, 50, 67, 1.3, "seam"),         # 51 x 68: the smallest taken a rectangle at a time
    (96, 40, 500, 3, 0.9, "seam"),
    (70, 70, 300, 200, 1.6, "smooth"),     # about 3,300 texels a tile: close to what LDS holds
    (70, 70, 300, 200, 1.8, "smooth"),     # more than that: scattered
    (64, 64, 211, 97, 1.0, "torn"),
    (64, 33, 100, 90, 1.0, "far"),
    (40, 40, 90, 90, 1.0, "none"),
    (700, 900, 3, 3, 0.01, "smooth"),      # more tiles than blocks
    (900, 700, 200, 300, 0.3, "seam"),
]


def gbuffer(W, H, tw, th, scale, kind, rng):
    y, x = np.mgrid[0:H, 0:W].astype(np.float64)
    u, v = (x * 0.97 + y * 0.11) * scale / tw, (y * 0.95 - x * 0.13) * scale / th
    if kind == "seam":
        u, v = (u + 0.98) % 1.0, (v + 0.97) % 1.0
    if kind == "torn":
        u, v = rng.random((H, W)), rng.random((H, W))
    if kind == "far":
        u, v = u * 3 - 40.3, v + 77.7
    n = np.stack([0.3 * np.sin(x / 9), 0.3 * np.cos(y / 7), np.ones_like(x)], -1)
    g = np.zeros((H, W, 12))
    g[..., 0:3], g[..., 3] = n, 1.0
    g[..., 4], g[..., 5], g[..., 6] = x / max(W, 1) - 0.5, y / max(H, 1) - 0.5, 0.1
    g[..., 8], g[..., 9] = u, v
    g[rng.random((H, W)) < (1.0 if kind == "none" else 0.1 if W > 1 else 0.0)] = 0.0
    return g.astype(np.float32)


def main():
    ctx = N.Context(64, 64)
    mesh = S.uv_sphere(6, 6, 1.0, tangents=True)
    for W, H, tw, th, scale, kind in CASES:
        print("[adjoint-tiles] %dx%d texture %dx%d %s" % (W, H, tw, th, kind), flush=True)
        rng = np.random.default_rng(W * 7 + tw)
        g = gbuffer(W, H, tw, th, scale, kind, rng)
        gb = A.GeometryBuffer(ctx, mesh, W, H, (0.0, 0.4, 3.0))
        gb.gbuf.copy_(torch.from_numpy(g))
        tex = rng.uniform(0.1, 0.9, (th, tw, 3)).astype(np.float32)
        gout = rng.uniform(0.1, 1.0, (H, W, 3)).astype(np.float32)
        t = torch.from_numpy(tex).cuda().requires_grad_()
        p = torch.tensor([0.9, 16.0], device="cuda").requires_grad_()
        out = A.shade(t, p, gb, 0.5)
        gt, gp = (v.cpu().numpy().astype(np.float64) for v in torch.autograd.grad(out, [t, p], torch.from_numpy(gout).cuda()))
        rt, rp = pyoracle.diff_backward_f64(g, tex, 0.9, 16.0, 0.5, gb.light.astype(np.float32),
                                            gb.eye.astype(np.float32), gout.astype(np.float64))
        err = lambda a, b: float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))  # noqa: E731
        print(json.dumps({"case": [W, H, tw, th, scale, kind], "tex": err(gt, rt),
                          "params": [err(gp[k], rp[k]) for k in range(2)]}), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
