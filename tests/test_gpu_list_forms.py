"""The list walks of the per-particle kernels at the sizes where they can go wrong, against the oracle,
bit for bit over three steps: a single particle, blocks that are not full, lists whose lengths leave
every remainder of four, walls on all sides (boundary lists longer than the fluid lists), and a
lattice without jitter, whose neighbors at exactly 2h make some blocks refuse the short gradient
factor and keep the exact one.
"""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend

import oracle_lib as O
from helpers import FIELDS_STEP, dam_break

pytestmark = pytest.mark.gpu

H = 0.01


@pytest.mark.parametrize("counts, jitter, layers", [((1, 1, 1), 0.01, 2), ((2, 1, 3), 0.01, 3), ((5, 7, 9), 0.01, 2),
                                                    ((4, 8, 8), 0.0, 2), ((16, 16, 16), 0.0, 2), ((33, 9, 17), 0.01, 3)])
def test_three_steps_match_the_oracle(counts, jitter, layers):
    print(f"case: {counts}, jitter {jitter}, {layers} wall layers", flush=True)
    tank = tuple(H * (c + 2) for c in counts)
    st = dam_break(counts[0], H, counts=counts, tank=tank, jitter_frac=jitter, layers=layers)
    p = scenes.make_params(H, termination_cond=scenes.TERM_POS)
    g = HipBackend(0)
    g.set_params(p)
    g.pull(st)
    o = O.Oracle(p, chunk_width=1, threads=4)
    o.pull(st)
    for s in range(3):
        g.step(1)
        o.step()
        assert g.info().solver_iters == o.info().solver_iters, s
    sg, so = g.push(), o.push()
    g.close()
    assert np.array_equal(sg.fluid_id, so.fluid_id)
    for f in FIELDS_STEP:
        assert np.array_equal(sg.fluid[f], so.fluid[f]), f
