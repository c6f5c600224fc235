"""Tiles of the adjoint's backward pass: edges of image tiles, textures kept in
LDS, taken a rectangle at a time and scattered, wrapping inside a tile, and
tiles without a covered pixel."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
def test_adjoint_tiles():
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "adjoint_tiles_check.py")], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    got = [json.loads(line) for line in r.stdout.splitlines() if line.startswith("{")]
    assert len(got) == 12
    for g in got:
        # FP32 sums of positive terms: far below 1e-5 of their sum; texture
        # coordinates far from 0 lose 2^-24 of their size (up to 120 texture
        # widths of 100 texels) in the weights
        assert g["tex"] <= (1e-3 if g["case"][5] == "far" else 1e-5), g
        assert max(g["params"]) <= (1e-3 if g["case"][5] == "far" else 1e-5), g
