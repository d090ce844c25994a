"""The rigid bodies' launches at the sizes where their form changes, against the oracle over three steps: a body
whose particles its own block updates (up to 2,048 in the context), one with more, one beyond the
one-block sort, and a fluid of so many blocks that the rigid queries take their turn on the stream. Lists
exact, fluid and body within 1e-5 (FP64 force sums in another order than the oracle's)."""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend

import oracle_lib as O
from helpers import rel_err

pytestmark = pytest.mark.gpu

H = 0.01


@pytest.mark.parametrize("fluid,side,nR", [(12, 0.15, (1000, 2048)), (12, 0.18, (2049, 16384)), (16, 0.5, (16385, 40000)),
                                           (65, 0.15, (1000, 2048))])
def test_three_steps_match_the_oracle(fluid, side, nR):
    print(f"case: {fluid}^3 fluid, cube of side {side}", flush=True)
    x = fluid * H + 0.5 * side + 0.005
    reach = max(fluid * H, side) + 0.1
    st = scenes.build_scene(scenes.rigid_cube_spec(fluid, H, side=side, center=(x, 0.5 * side + 0.02, 0.5 * side + 0.02),
                                                   tank=(x + 0.5 * side + 0.1, reach, reach)))
    assert nR[0] <= st.n[2] <= nR[1] and st.n[3] == 1
    p = scenes.make_params(H, termination_cond=scenes.TERM_POS)
    g = HipBackend(0)
    g.set_params(p)
    g.pull(st)
    o = O.Oracle(p, chunk_width=1)
    o.pull(st)
    for s in range(3):
        g.step(1)
        o.step()
        assert g.info().solver_iters == o.info().solver_iters, s
    for rel in (O.FR, O.RF):
        cg, ig = g.neighbors(rel)
        co, io, _ = o.lists(rel)
        assert co.sum() > 0
        assert np.array_equal(cg, co) and np.array_equal(ig, io)
    sg, so = g.push(), o.push()
    assert np.array_equal(sg.fluid_id, so.fluid_id)
    for f in ("x", "y", "z", "vx", "vy", "vz", "density", "pressure"):
        assert rel_err(sg.fluid[f], so.fluid[f]) <= 1e-5, f
    for f in ("xcm", "ycm", "zcm", "vx", "vy", "vz", "wx", "wy", "wz", "a00", "a11", "a22", "a01"):
        assert rel_err(sg.body[f], so.body[f]) <= 1e-5, f
    xg, vg = g.rigid_world()
    xo, vo = o.rigid_world()
    assert rel_err(xg, xo) <= 1e-6
    assert rel_err(vg, vo) <= 1e-5
