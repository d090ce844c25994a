"""The pressure solve in one launch (contexts of up to one 256-particle block per CU) against the same solve
launch by launch (a profiled context), every field after every step bit for bit, and the solver's report:
one block, a block that is not full, one block per CU and one more, every termination condition and the
warm start, lists longer than a thread keeps (compressed fluid; walls of three layers in a corner), blocks
without a halo (the most compressed), a rigid body, and several scenes that stop at different sweeps in one context."""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend, HipBatch

from helpers import FIELDS_STEP, dam_break

pytestmark = pytest.mark.gpu

H = 0.01


def squeezed(factor):
    """a block whose lattice is closer than the particle size: more FF entries than a thread keeps"""
    st = dam_break(18, H, tank=(0.3, 0.2, 0.2))
    for f in "xyz":
        st.fluid[f][:] = (st.fluid[f] - np.float32(0.5 * H)) * np.float32(factor) + np.float32(0.5 * H)
    return st


def block(nx, ny, nz, **kw):
    return dam_break(nx, H, counts=(nx, ny, nz), tank=(H * (nx + 8), H * (ny + 8), H * (nz + 8)), **kw)


SCENES = {
    "one block": (lambda: block(6, 6, 7), {}),
    "not full": (lambda: block(13, 9, 11), dict(termination_cond=scenes.TERM_ABS)),
    "256 blocks": (lambda: block(64, 32, 32), dict(jacobi_warm_start=0.5)),
    "257 blocks": (lambda: block(65, 32, 32), {}),
    "fixed": (lambda: block(30, 20, 20), dict(termination_cond=scenes.TERM_FIXED)),
    "raw": (lambda: block(30, 20, 20), dict(termination_cond=scenes.TERM_RAW)),
    "squeezed": (lambda: squeezed(0.9), {}),
    "squeezed more": (lambda: squeezed(0.75), dict(termination_cond=scenes.TERM_FIXED)),
    "corner": (lambda: dam_break(12, H, counts=(12, 12, 12), tank=(0.13, 0.13, 0.13), layers=3), {}),
    "rigid": (lambda: scenes.build_scene(scenes.rigid_cube_spec(16, H, side=0.06, center=(0.25, 0.1, 0.15), tank=(0.4, 0.3, 0.3))), {}),
}


def same(a, b):
    assert np.array_equal(a.fluid_id, b.fluid_id)
    for f in FIELDS_STEP:
        assert np.array_equal(a.fluid[f], b.fluid[f], equal_nan=True), f
    for f in a.body:
        assert np.array_equal(a.body[f], b.body[f], equal_nan=True), f


def same_report(a, b):
    for f in ("solver_iters", "sweeps_total", "avg_err_raw", "avg_err_pos", "avg_err_abs", "err_sum_raw", "err_sum_pos", "err_sum_abs",
              "flags"):
        assert getattr(a, f) == getattr(b, f), f


@pytest.mark.parametrize("name", SCENES)
def test_one_launch_equals_launch_by_launch(name):
    print(f"case: {name}", flush=True)
    make, kw = SCENES[name]
    st = make()
    p = scenes.make_params(H, **{"termination_cond": scenes.TERM_POS, **kw})
    runs = []
    for timed in (False, True):
        g = HipBackend(0)
        g.set_params(p)
        g.profile_enable(timed)
        g.pull(st)
        runs.append(g)
    for _ in range(3):
        for g in runs:
            g.step(1)
        same(runs[0].push(), runs[1].push())
        same_report(runs[0].info(), runs[1].info())


def test_scenes_of_one_context_stop_by_themselves():
    print("case: four scenes in one context", flush=True)
    cases = [(block(9, 9, 9), scenes.TERM_POS), (block(21, 17, 13), scenes.TERM_ABS), (block(16, 16, 16), scenes.TERM_FIXED),
             (squeezed(0.9), scenes.TERM_POS)]
    specs = [(scenes.make_params(H, termination_cond=t), st) for st, t in cases]
    b = HipBatch(0)
    ids = b.update(add=specs)
    alone = []
    for p, st in specs:
        g = HipBackend(0)
        g.set_params(p)
        g.profile_enable(True)
        g.pull(st)
        alone.append(g)
    for _ in range(3):
        b.step(1)
        for i, g in zip(ids, alone):
            g.step(1)
            same(b.push(i), g.push())
            same_report(b.info(i), g.info())


def test_context_that_held_a_larger_scene():
    print("case: 120,000 particles, then 4,900, then 65,000", flush=True)
    p = scenes.make_params(H, termination_cond=scenes.TERM_POS)
    g = HipBackend(0)
    g.set_params(p)
    for st in (block(60, 50, 40), block(17, 17, 17), block(65, 40, 25)):
        fresh = HipBackend(0)
        fresh.set_params(p)
        fresh.profile_enable(True)
        for b in (g, fresh):
            b.pull(st)
            b.step(2)
        same(g.push(), fresh.push())
        same_report(g.info(), fresh.info())
        if st.n[0] < 65536:
            # the solve's records are sized by the scene, not by the pools that the context keeps
            assert g.memory().alloc_bytes - fresh.memory().alloc_bytes < (1 << 30)
