"""Backward pass of the adjoint on images of few pixels: the edges of its 8 x 8
and 16 x 16 squares, textures of one texel to a million, pixels that all share
texels or none do, the sizes where it gives way to image tiles, and tiles from
there on.  Run in a process of its own by tests/test_adjoint_small.py (torch
must be imported before libpsgpu loads).  Prints one JSON line per case (see
adjoint_tiles_check.py), and one with the kernel's time in us on two images."""
import ctypes as C
import json

import torch

import adjoint_tiles_check as T
from puresoft3d_amd import adjoint as A
from puresoft3d_amd import native as N
from puresoft3d_amd import scenes as S

CASES = [
    (1, 1, 300, 200, 1.0, "smooth"),
    (32, 32, 1, 1, 0.01, "smooth"),        # every texel of a footprint is the same one
    (17, 15, 2, 1, 0.1, "seam"),
    (15, 17, 50, 67, 1.1, "seam"),
    (33, 31, 1, 40, 0.3, "seam"),
    (50, 50, 8, 8, 0.1, "smooth"),         # 2,500 pixels, 64 texels: the last of them here
    (51, 51, 8, 8, 0.1, "smooth"),         # and the first in tiles
    (64, 64, 1024, 1024, 0.01, "smooth"),  # a wave's pixels in one texel
    (257, 127, 211, 97, 1.0, "torn"),
    (181, 140, 250, 130, 1.3, "smooth"),
    (65, 63, 90, 90, 0.5, "none"),
    (70, 33, 100, 90, 1.0, "far"),
    (4096, 8, 90, 70, 0.5, "seam"),        # 32,768 pixels: the last of them here
    (9, 3641, 90, 70, 0.5, "seam"),        # and the first in tiles
    (257, 129, 49, 67, 1.1, "seam"),       # as in adjoint_tiles_check.py, above that size
    (257, 129, 50, 67, 1.3, "seam"),
    (225, 160, 300, 200, 1.6, "smooth"),
    (225, 160, 300, 200, 1.8, "smooth"),
    (33, 1025, 211, 97, 1.0, "torn"),
    (257, 129, 90, 90, 1.0, "none"),
]


def microseconds(ctx, size, tw, th):
    gb = A.GeometryBuffer(ctx, S.uv_sphere(60, 60, 1.0, tangents=True), size, size, (0.0, 0.4, 3.0))
    tex, out = torch.rand((th, tw, 3), device="cuda"), torch.rand((size, size, 3), device="cuda")
    par = torch.tensor([0.9, 16.0], device="cuda")
    gt, gp = torch.zeros_like(tex), torch.zeros_like(par)
    d, p = gb.desc(tex, 0.5), lambda t: C.c_void_p(t.data_ptr())

    def call():
        rc = N.lib().psgpu_diff_backward(ctx.h, C.byref(d), p(gb.gbuf), p(tex), p(par), p(out), p(gt), p(gp), A._stream())
        assert rc == 0
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(20):
            call()
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    best = 1e9
    for _ in range(7):
        a.record()
        graph.replay()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / 20)
    return best


def main():
    T.CASES[:] = CASES
    T.main()
    print("[adjoint-small] times", flush=True)
    ctx = N.Context(64, 64)
    print(json.dumps({"us": [microseconds(ctx, size, 250, 130) for size in (64, 512)]}), flush=True)
    ctx.close()


if __name__ == "__main__":
    main()
