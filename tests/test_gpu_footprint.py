"""tsp_batch_footprint against the memory that a context of one scene holds: at least what it holds besides its
cell tables, at sizes around the limit of the one-launch solve, and in a context that held a larger scene."""
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend, HipBatch

pytestmark = pytest.mark.gpu

H = 0.01


def held(g):
    """bytes in use without the cell tables (24 bytes per cell of the frame)"""
    g.trim()
    d = g.info().frame_dim
    return g.memory().alloc_bytes - 24 * d[0] * d[1] * d[2]


def spec(counts):
    return scenes.dam_break_spec(counts[0], H, counts=counts, tank=tuple((c + 8) * H for c in counts))


def backend():
    g = HipBackend(0)
    g.set_params(scenes.make_params(H, termination_cond=scenes.TERM_POS))
    return g


@pytest.mark.parametrize("counts", [(6, 6, 7), (17, 16, 16), (40, 40, 40), (64, 32, 32), (257, 16, 16), (61, 37, 49)])
def test_footprint_covers_the_scene(counts):
    print(f"case: {counts}", flush=True)
    g = backend()
    g.pull_spec(spec(counts))
    g.step(2)
    foot = HipBatch.footprint(g.n)
    print(held(g), foot, flush=True)
    assert held(g) <= foot


def test_records_of_the_solve_follow_the_scene():
    # the list pools are kept, so a context that held a larger scene holds more than a fresh one; the
    # solve's wall records are the scene's own
    print("case: 30,000 particles in a context that held 216,000", flush=True)
    fresh, g = backend(), backend()
    big, small = spec((60, 60, 60)), spec((31, 31, 31))
    for b, specs in ((fresh, [small]), (g, [big, small])):
        for s in specs:
            b.pull_spec(s)
            b.step(1)
    # (the pools of 216,000 particles: 80 entries of 2 bytes each, and their growth by an eighth)
    pools = 160 * 216_000 * 9 // 8 + (1 << 20)
    assert held(g) - held(fresh) <= pools
