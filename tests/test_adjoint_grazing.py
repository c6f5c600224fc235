"""The highlights that the image has are those that the gradients have, also
where the half vector grazes the surface."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.gpu
def test_grazing_highlights():
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "adjoint_grazing_check.py")], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-3000:]
    got = [json.loads(line) for line in r.stdout.splitlines() if line.startswith("{")]
    assert len(got) == 2
    for g in got:
        assert 0.3 < g["facing"] < 0.7, g
        # s is rounded once (2^-24 of it), its power with 0.05 and logarithm
        # are a few ulp, and the sums' terms have one sign: far below 1e-5.  A
        # highlight of the wrong sign of s is 0.2 of the largest colour.
        assert g["image"] <= 1e-5, g
        assert g["exponent"] <= 1e-5, g
