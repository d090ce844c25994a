"""The short forms of the pair kernels (rootRcp, kgFactor<true>, kgShort with its stored correction,
in tsp_device.h) against the general correctly rounded lowering, bit for bit and exhaustively, on
the GPU: tests/cpp/pair_selftest.hip, built into turbospharticles_amd/lib/.
"""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_short_root_and_gradient_factor_match_the_general_lowering():
    print("case: pair_selftest (roots exhaustive, gradient factors over the support)", flush=True)
    exe = os.path.join(ROOT, "turbospharticles_amd", "lib", "pair_selftest")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "PASS" in r.stdout
