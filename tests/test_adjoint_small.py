"""The adjoint's backward pass on images of few pixels, and at the sizes where
it changes to image tiles."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
def test_adjoint_small():
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "adjoint_small_check.py")], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    lines = [json.loads(line) for line in r.stdout.splitlines() if line.startswith("{")]
    got = [g for g in lines if "case" in g]
    assert len(got) == 20
    for g in got:
        # FP32 sums of positive terms, at most some 1,000 of them by turns:
        # far below 1e-5 of their sum; coordinates of up to 120 texture widths
        # of 100 texels lose 2^-24 of their size in the weights
        far = g["case"][5] == "far"
        assert g["tex"] <= (1e-3 if far else 1e-5), g
        assert max(g["params"]) <= (1e-3 if far else 1e-5), g
    # 64 x 64 pixels are a 64th of 512 x 512; in four tiles they took longer
    small, large = lines[-1]["us"]
    assert small < 0.6 * large, lines[-1]
