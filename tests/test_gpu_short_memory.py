"""Calls that find no device memory (a memory limit stands for the full GPU): each fails with an error and
leaves a context that refuses or goes on, and once there is memory gives the bits of one that never ran short."""
import numpy as np
import pytest

from turbospharticles_amd import scenes
from turbospharticles_amd.backend import HipBackend, HipBatch, TspError

from helpers import FIELDS_STEP, cube_scene, dam_break

pytestmark = pytest.mark.gpu

H = 0.01
TSP_ERR_HIP, TSP_ERR_STATE = -2, -3
NO_LIMIT = (1 << 64) - 1
PARAMS = scenes.make_params(H, termination_cond=scenes.TERM_POS)


def backend():
    g = HipBackend(0)
    g.set_params(PARAMS)
    return g


def same(a, b):
    assert np.array_equal(a.fluid_id, b.fluid_id)
    for f in FIELDS_STEP:
        assert np.array_equal(a.fluid[f], b.fluid[f]), f
    for f in a.body:
        assert np.array_equal(a.body[f], b.body[f]), f


def squeezed(factor):
    st = dam_break(18, H, tank=(0.3, 0.2, 0.2))
    for f in "xyz":
        st.fluid[f][:] = (st.fluid[f] - np.float32(0.5 * H)) * np.float32(factor) + np.float32(0.5 * H)
    return st


def whole(g, st):
    """what a program does with a scene, from the pull to the export"""
    g.pull(st)
    g.step(2)
    stats = g.statistics()
    snap = g.export_snapshot()
    return g.push(), snap, list(stats.nbr_avg)


@pytest.mark.parametrize("case", ["dam", "contact", "squeezed"])
def test_every_allocation_may_fail(case):
    # the limit rises from nothing in small steps, so that each attempt ends at a later allocation
    print(f"case: {case}", flush=True)
    st = {"dam": lambda: dam_break(14, H), "contact": lambda: cube_scene(center=(0.15, 0.031, 0.15), vel=(0.0, -0.5, 0.0)),
          "squeezed": lambda: squeezed(0.75)}[case]()
    ref = backend()
    want, want_snap, want_avg = whole(ref, st)
    ref.trim()
    need = ref.memory().alloc_bytes
    ref.close()
    g = backend()
    g.n = st.n   # (the calls below reach the library before the first pull succeeds, too)
    failed = []
    for k in range(1, 200):
        g.set_memory_limit(need * k // 40)
        try:
            got, snap, avg = whole(g, st)
            break
        except TspError as e:
            assert e.code == TSP_ERR_HIP, e
            failed.append(k)
            # whatever failed, further calls answer or refuse
            for call in (lambda: g.step(1), g.neighbor_search, g.statistics, g.sort_state, g.export_snapshot,
                         lambda: g.neighbors(0), lambda: g.set_params(PARAMS), g.push, g.info):
                try:
                    call()
                except TspError as e2:
                    assert e2.code in (TSP_ERR_HIP, TSP_ERR_STATE), e2
    print("limits that refused:", failed, flush=True)
    assert len(failed) >= 20
    same(got, want)
    assert np.array_equal(snap.fluid_xyz, want_snap.fluid_xyz) and avg == want_avg


def test_a_pool_that_cannot_grow():
    print("case: the list pools cannot grow, then can", flush=True)
    st = squeezed(0.75)
    ref, g = backend(), backend()
    for b in (ref, g):
        b.pull(st)
    ref.step(3)
    for b in (ref, g):
        b.trim()
    g.set_memory_limit(ref.memory().alloc_bytes + g.memory().alloc_bytes)
    for _ in range(2):
        with pytest.raises(TspError) as e:
            g.step(1)
        assert e.value.code == TSP_ERR_HIP
        with pytest.raises(TspError) as e:
            g.export_snapshot()
        assert e.value.code == TSP_ERR_STATE
    g.set_memory_limit(NO_LIMIT)
    g.step(3)
    same(g.push(), ref.push())


def test_an_admission_without_memory_leaves_the_residents():
    print("case: scenes that do not fit beside resident ones", flush=True)
    a, big = dam_break(12, H), dam_break(40, H)
    ref = backend()
    ref.pull(a)
    ref.step(4)
    b = HipBatch(0)
    sid = b.add(PARAMS, a)
    b.step(1)
    b.trim()
    ref.trim()
    base = ref.memory().alloc_bytes + b.memory().alloc_bytes
    # from too little for the new arena to too little for the last buffers behind it
    need = HipBatch.footprint(big.n)
    refused = 0
    for part in range(1, 13):
        b.set_memory_limit(base + need * part // 12)
        try:
            new = b.update(add=[(PARAMS, big)])
            b.set_memory_limit(NO_LIMIT)
            b.update(remove=new)
            break
        except TspError as e:
            assert e.code == TSP_ERR_HIP, e
            refused += 1
            assert b.ids() == [sid]
    print("refused:", refused, flush=True)
    assert refused >= 4
    b.set_memory_limit(NO_LIMIT)
    b.step(3)
    same(b.push(sid), ref.push())
