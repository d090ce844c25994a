"""Which form a solve takes, and the way out of the one-launch form: a scene whose blocks do not all come to the
entry is given up before anything is written, and the step is finished launch by launch with the same bits; the next
256 steps do not try again."""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend, HipBatch

from helpers import FIELDS_STEP, dam_break

pytestmark = pytest.mark.gpu

H = 0.01
HOLD = 256


def block(nx, ny, nz, **kw):
    return dam_break(nx, H, counts=(nx, ny, nz), tank=(H * (nx + 8), H * (ny + 8), H * (nz + 8)), **kw)


def cube():
    return scenes.build_scene(scenes.rigid_cube_spec(16, H, side=0.06, center=(0.25, 0.1, 0.15), tank=(0.4, 0.3, 0.3)))


def params(term):
    return scenes.make_params(H, termination_cond=term)


def backend(st, term=scenes.TERM_POS, timed=False):
    g = HipBackend(0)
    g.set_params(params(term))
    g.profile_enable(timed)   # (timed launches: the sweeps launch by launch)
    g.pull(st)
    return g


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


@pytest.mark.parametrize("counts, one", [((6, 6, 7), True), ((16, 16, 16), True), ((17, 16, 16), True), ((64, 32, 32), True),
                                         ((257, 16, 16), False), ((61, 37, 49), False)])
def test_form_by_the_number_of_blocks(counts, one):
    # 1, 16, 17, 256, 257 and 433 blocks
    print(f"case: {counts}", flush=True)
    g = backend(block(*counts))
    g.step(3)
    assert g.solve_forms() == ((3, 0, 0) if one else (0, 0, 3))
    timed = backend(block(*counts), timed=True)
    timed.step(3)
    assert timed.solve_forms() == (0, 0, 3)
    same(g.push(), timed.push())
    same_report(g.info(), timed.info())


def test_walls_that_need_longer_records():
    # 250 particles in a tube one particle wide: more than the 16 wall entries per slot (and 1,024) that the
    # records have room for to begin with
    print("case: 250 particles in a tube", flush=True)
    st = dam_break(250, H, counts=(250, 1, 1), tank=(2.51, 0.01, 0.01))
    g, timed = backend(st), backend(st, timed=True)
    for b in (g, timed):
        b.step(3)
    assert g.info().n_fb > 16 * 256 + 1024
    assert g.solve_forms() == (3, 0, 0)
    same(g.push(), timed.push())
    same_report(g.info(), timed.info())


@pytest.mark.parametrize("name", ["one block", "not full", "256 blocks", "body", "abs"])
def test_given_up_scene_is_solved_launch_by_launch(name):
    print(f"case: {name}", flush=True)
    st = {"one block": lambda: block(6, 6, 7), "not full": lambda: block(13, 9, 11), "256 blocks": lambda: block(64, 32, 32),
          "body": cube, "abs": lambda: block(16, 16, 16)}[name]()
    term = scenes.TERM_ABS if name == "abs" else scenes.TERM_POS
    g, timed = backend(st, term), backend(st, term, timed=True)
    g.step(1)
    g.hold_solve()
    for b, n in ((g, 1), (timed, 2)):
        b.step(n)
    assert g.solve_forms() == (1, 1, 0)
    same(g.push(), timed.push())
    same_report(g.info(), timed.info())
    for b in (g, timed):
        b.step(2)
    assert g.solve_forms() == (1, 1, 2)
    same(g.push(), timed.push())
    same_report(g.info(), timed.info())


def test_the_form_is_tried_again():
    print("case: 256 steps after a solve that was given up", flush=True)
    st = block(8, 8, 8)
    g, timed = backend(st, scenes.TERM_FIXED), backend(st, scenes.TERM_FIXED, timed=True)
    g.hold_solve()
    g.step(1 + HOLD)
    assert g.solve_forms() == (0, 1, HOLD)
    g.step(1)
    assert g.solve_forms() == (1, 1, HOLD)
    timed.step(2 + HOLD)
    same(g.push(), timed.push())


@pytest.mark.parametrize("held", [0, 1, 2, 3])
def test_one_scene_of_a_context_is_given_up(held):
    # the others converge in the one launch (after different numbers of sweeps), the held one in launches after it
    print(f"case: four scenes, scene {held} held at the entry", flush=True)
    cases = [(block(9, 9, 9), scenes.TERM_POS), (block(21, 17, 13), scenes.TERM_ABS), (cube(), scenes.TERM_POS),
             (block(16, 16, 16), scenes.TERM_FIXED)]
    b = HipBatch(0)
    ids = b.update(add=[(params(t), st) for st, t in cases])
    alone = [backend(st, t, timed=True) for st, t in cases]
    b.step(1)
    b.hold_solve(ids[held])
    b.step(1)
    assert b.solve_forms() == (1, 1, 0)
    for g in alone:
        g.step(2)
    for _ in range(2):
        for i, g in zip(ids, alone):
            same(b.push(i), g.push())
            same_report(b.info(i), g.info())
        b.step(1)
        for g in alone:
            g.step(1)
    assert b.solve_forms() == (1, 1, 2)
