"""Both passes of the adjoint where the half vector grazes the surface: normals
within some 1e-7 of perpendicular to it, half of them facing it, and a small
exponent, so that a highlight is a large term or none.  Run in a process of
its own by tests/test_adjoint_grazing.py (torch must be imported before
libpsgpu loads).  Prints one JSON line: the relative errors of the image and
of the exponent's gradient against the FP64 oracle."""
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


def main():
    ctx = N.Context(64, 64)
    rng = np.random.default_rng(17)
    for W, H in ((64, 48), (300, 200)):
        print("[adjoint-grazing] %dx%d" % (W, H), flush=True)
        gb = A.GeometryBuffer(ctx, S.uv_sphere(6, 6, 1.0, tangents=True), W, H, (0.0, 0.4, 3.0))
        unit = lambda v: v / np.linalg.norm(v, axis=-1, keepdims=True)  # noqa: E731
        at = rng.uniform(-0.5, 0.5, (H, W, 3)).astype(np.float32).astype(np.float64)
        light, eye = gb.light.astype(np.float32).astype(np.float64), gb.eye.astype(np.float32).astype(np.float64)
        half = unit(unit(light - at) + unit(eye - at))
        side = unit(np.cross(half, unit(rng.normal(size=(H, W, 3)))))
        g = np.zeros((H, W, 12), np.float32)
        g[..., 0:3] = side + rng.uniform(-1e-7, 1e-7, (H, W, 1)) * half
        g[..., 3] = 1.0
        g[..., 4:7] = at
        g[..., 8:10] = rng.random((H, W, 2))
        s = (unit(g[..., 0:3].astype(np.float64)) * half).sum(-1)
        gb.gbuf.copy_(torch.from_numpy(g))
        tex = rng.uniform(0.1, 0.9, (5, 7, 3)).astype(np.float32)
        gout = rng.uniform(0.1, 1.0, (H, W, 3)).astype(np.float32)
        t = torch.from_numpy(tex).cuda().requires_grad_()
        p = torch.tensor([0.9, 0.05], device="cuda").requires_grad_()
        out = A.shade(t, p, gb, 0.5)
        gp = torch.autograd.grad(out, p, torch.from_numpy(gout).cuda())[0].cpu().numpy().astype(np.float64)
        exponent = float(np.float32(0.05))
        lights = (gb.light.astype(np.float32), gb.eye.astype(np.float32))
        ref = pyoracle.diff_forward_f64(g, tex, float(np.float32(0.9)), exponent, 0.5, *lights)
        _, rp = pyoracle.diff_backward_f64(g, tex, float(np.float32(0.9)), exponent, 0.5, *lights, gout.astype(np.float64))
        image = np.abs(out.detach().cpu().numpy() - ref).max() / np.abs(ref).max()
        print(json.dumps({"size": [W, H], "facing": float((s > 0).mean()), "image": float(image),
                          "exponent": float(abs(gp[1] - rp[1]) / abs(rp[1]))}), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
