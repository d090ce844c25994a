"""The device blocks that a context keeps of a replaced layout: counted in the memory report, bounded over
all contexts of a GPU, given back on trim, and given back when another context has no other memory."""
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend, TspError

pytestmark = pytest.mark.gpu

H = 0.01
MOST, MOST_ON_DEVICE = 2 << 30, 8 << 30
TSP_ERR_HIP = -2


def backend():
    g = HipBackend(0)
    g.set_params(scenes.make_params(H, termination_cond=scenes.TERM_POS))
    return g


def spec(side):
    return scenes.dam_break_spec(side, H, tank=tuple(r * side * H for r in scenes.TANK_RATIO))


def held(g):
    m = g.memory()
    assert m.alloc_bytes == sum(m.particles) + sum(m.search) + sum(m.lists) + m.misc
    assert m.peak_alloc_bytes >= m.alloc_bytes
    return m.alloc_bytes


def trimmed(g):
    """what is in use after the kept blocks went, and how much they were"""
    before = held(g)
    g.trim()
    return held(g), before - held(g)


def test_kept_blocks_are_counted_and_trimmed():
    print("case: 100,000 particles, then 8,000", flush=True)
    g = backend()
    g.pull_spec(spec(46))
    in_use, _ = trimmed(g)
    g.pull_spec(spec(20))
    # the replaced arena is kept: at least the 160 bytes of records per particle
    small, kept = trimmed(g)
    assert kept >= 160 * 46 ** 3
    assert small < in_use
    assert trimmed(g) == (small, 0)
    g.step(2)
    assert g.info().step == 2


def test_another_context_takes_what_one_keeps():
    print("case: kept blocks of one context, a second context that needs their memory", flush=True)
    a, b = backend(), backend()
    a.pull_spec(spec(60))
    a.pull_spec(spec(16))
    b.pull_spec(spec(40))
    need, _ = trimmed(b)
    b.close()
    kept_a = held(a)
    b = backend()
    # room for both scenes, not for a's kept blocks besides
    b.set_memory_limit(kept_a + need // 2)
    assert need > 0 and kept_a > 2 * need
    b.pull_spec(spec(40))
    b.step(1)
    assert held(a) < kept_a
    assert trimmed(a)[1] == 0
    # and a limit that no give-back can meet refuses, and leaves both contexts as they are
    b.set_memory_limit(held(a) + held(b))
    with pytest.raises(TspError) as e:
        b.pull_spec(spec(60))
    assert e.value.code == TSP_ERR_HIP
    a.step(1)
    assert a.info().step == 1


def test_contexts_keep_no_more_than_the_bounds():
    print("case: six contexts that replace 8,000,000 particles", flush=True)
    runs = [backend() for _ in range(6)]
    for g in runs:
        g.pull_spec(spec(200))
        g.pull_spec(spec(16))
    kept = [trimmed(g)[1] for g in runs]
    print(kept, flush=True)
    assert max(kept) <= MOST and 2 * MOST < sum(kept) <= MOST_ON_DEVICE
