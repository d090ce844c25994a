"""The quotient of the pair kernels as they run it (quotFrom with rootRcp's estimate, kgFactor<true>,
kgShort with its correction, in tsp_device.h) against the general correctly rounded lowering.

On its own over the whole range of operands that the host allows, with every numerator for the distances
next to a power of two (tests/cpp/quotient_selftest.hip, built into turbospharticles_amd/lib/), and in a step:
particle sizes whose gradient scale meets a distance just below a power of two, where the quotient lies
2^-25 of an ulp from a midpoint, must match the oracle bit for bit."""
import os
import subprocess

import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend

import oracle_lib as O
from helpers import FIELDS_STEP

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_quotient_from_the_reciprocal_root_matches_the_general_lowering():
    print("case: quotient_selftest (random pairs over the allowed range, every numerator at the critical distances, "
          "outer branch at 50 particle sizes)", flush=True)
    exe = os.path.join(ROOT, "turbospharticles_amd", "lib", "quotient_selftest")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "PASS" in r.stdout


# the particle size and the distance's mantissa below 2^-6 (in units of 2^-30); the first pair is the closest case
# (koutScale's mantissa is 0x7ffffe), the others lie beside it
@pytest.mark.parametrize("h, below", [(0.013813708, 1), (0.013813708, 2), (0.013813708, 3), (0.013813709, 1), (0.01, 1)])
def test_pair_whose_quotient_is_nearly_a_midpoint(h, below):
    print(f"case: h = {h}, distance 2^-6 - {below} * 2^-30, one step", flush=True)
    h = float(np.float32(h))
    st = scenes.build_scene(scenes.dam_break_spec(0, h, counts=(3, 3, 3), tank=(0.2, 0.2, 0.2)))
    f, b = st.fluid, st.boundary
    anchor = np.array([f[a][0] for a in "xyz"], np.float32)
    for arr in (f, b):
        for a, key in enumerate("xyz"):
            arr[key][:] = arr[key] - anchor[a]
    st.domain = (st.domain[0] - anchor, st.domain[1] - anchor)
    dist = np.float32(2.0 ** -6 - below * 2.0 ** -30)
    f["x"][1], f["y"][1], f["z"][1] = dist, np.float32(0.0), np.float32(0.0)
    f["vx"][1], f["vx"][0] = np.float32(-0.7), np.float32(0.3)
    p = scenes.make_params(h, termination_cond=scenes.TERM_POS)
    g, o = HipBackend(0), O.Oracle(p, chunk_width=1, threads=8)
    g.set_params(p)
    for s in (g, o):
        s.pull(st)
    g.step(1)
    o.step()
    sg, so = g.push(), o.push()
    assert np.array_equal(sg.fluid_id, so.fluid_id)
    for fld in FIELDS_STEP:
        assert np.array_equal(sg.fluid[fld], so.fluid[fld]), fld
