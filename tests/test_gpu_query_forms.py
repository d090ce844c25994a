"""The neighbor query's walks at the forms where they can go wrong, every list of the oracle entry by entry,
then one step bit for bit:

  - frames of other cell sizes: wide cells (rows of more than 32 candidates, which the hit masks do not
    cover), narrow cells (a stencil of more than three cells per axis);
  - particles on a coordinate plane (pairs may be nearer than 2^-48: the walk that looks for them) and
    walls in the same place;
  - sparse particles above a dense bed (blocks whose neighbors lie in many pages: no halo), and blocks of
    both;
  - particles outside the domain and the frame;
  - more blocks than one launch shares per particle (kShareBlocks), and one more than that.
"""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend

import oracle_lib as O
from helpers import FIELDS_STEP, dam_break

pytestmark = pytest.mark.gpu

H = 0.01


def shifted(st, by):
    """the scene moved by a vector (positions and domain)"""
    for a, f in enumerate("xyz"):
        st.fluid[f] += np.float32(by[a])
        st.boundary[f] += np.float32(by[a])
    st.domain = tuple(d + np.float32(by) for d in st.domain)
    return st


def spray():
    """a bed of 96 x 8 x 96 particles with single ones 4 h apart above it"""
    st = dam_break(96, H, counts=(96, 9, 96), tank=(1.2, 0.6, 1.2))
    top = st.fluid["y"] > 8 * H
    ix, iz = (np.floor(st.fluid[f] / np.float32(H)).astype(int) for f in "xz")
    # particles of the top layer that stay sit 4 h apart; the others go up, as far from each other
    stay = top & (ix % 4 == 0) & (iz % 4 == 0)
    rest = np.flatnonzero(top & ~stay)
    st.fluid["y"][rest] += np.float32(H) * (3 + 4 * (np.arange(rest.size) % 7)).astype(np.float32)
    return st


def stray():
    st = dam_break(20, H, tank=(0.5, 0.3, 0.3))
    for k, (x, y, z) in enumerate([(-0.4, 0.1, 0.1), (0.2, 0.9, 0.1), (0.201, 0.9, 0.1), (2.0, 2.0, 2.0), (0.1, 0.1, -0.09)]):
        st.fluid["x"][k], st.fluid["y"][k], st.fluid["z"][k] = x, y, z
    return st


CASES = {
    "ratio 0.4": (lambda: dam_break(14, H, tank=(0.3, 0.2, 0.2)), dict(grid_cell_size_ratio=0.4)),
    "ratio 0.6": (lambda: dam_break(18, H, tank=(0.3, 0.2, 0.2)), dict(grid_cell_size_ratio=0.6)),
    "ratio 1.3": (lambda: dam_break(18, H, tank=(0.3, 0.2, 0.2)), dict(grid_cell_size_ratio=1.3)),
    "ratio 2.5": (lambda: dam_break(18, H, tank=(0.3, 0.2, 0.2)), dict(grid_cell_size_ratio=2.5)),
    "on a plane": (lambda: shifted(dam_break(17, H, tank=(0.3, 0.2, 0.2), jitter_frac=0.0), (-0.5 * H, 0.0, -7.5 * H)), {}),
    "spray": (spray, {}),
    "stray": (stray, {}),
    "512 blocks": (lambda: dam_break(64, H, counts=(64, 32, 64), tank=(0.8, 0.5, 0.8)), {}),
    "513 blocks": (lambda: dam_break(64, H, counts=(64, 32, 65), tank=(0.8, 0.5, 0.8)), {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_lists_and_one_step_match_the_oracle(name):
    print(f"case: {name}", flush=True)
    make, kw = CASES[name]
    st = make()
    p = scenes.make_params(H, termination_cond=scenes.TERM_FIXED, **kw)
    g = HipBackend(0)
    g.set_params(p)
    g.pull(st)
    o = O.Oracle(p, chunk_width=1, threads=8)
    o.pull(st)
    g.neighbor_search()
    o.neighbor_search()
    for rel in (O.FF, O.FB, O.FR):
        cg, ig = g.neighbors(rel)
        co, io, _ = o.lists(rel)
        assert np.array_equal(cg, co), rel
        assert np.array_equal(ig, io), rel
    g.step(1)
    o.step()
    sg, so = g.push(), o.push()
    g.close()
    assert np.array_equal(sg.fluid_id, so.fluid_id)
    for f in FIELDS_STEP:
        assert np.array_equal(sg.fluid[f], so.fluid[f]), f
