"""State fields between the caller's arrays and the device records, bit for bit: sizes around a thread
block's words and around the staging buffers, populations that are empty, several scenes in one update and
fields that a view leaves out."""
import ctypes

import numpy as np
import pytest

from turbospharticles_amd import _capi, scenes
from turbospharticles_amd.backend import HipBackend, HipBatch

pytestmark = pytest.mark.gpu


def random_state(n, seed):
    """every field of its own random bits of finite floats; positions inside the unit box"""
    rng = np.random.default_rng(seed)
    st = _capi.HostState(*n)
    for group in (st.fluid, st.boundary, st.rigid, st.body):
        for k, f in group.items():
            f[:] = rng.random(f.size, np.float32) * (0.9 if k in "xyz" else 1e3) + 0.01
    st.fluid_id[:] = rng.integers(0, 2 ** 63, n[0], np.uint64)
    st.boundary_id[:] = rng.integers(0, 2 ** 63, n[1], np.uint64)
    st.rigid_id[:] = rng.integers(0, 2 ** 63, n[2], np.uint64)
    if n[3]:
        st.rigid_body[:] = np.sort(rng.integers(0, n[3], n[2]))
        st.body_id[:] = rng.integers(0, 2 ** 31, n[3])
        st.body_count[:] = np.bincount(st.rigid_body, minlength=n[3])
    st.domain = (np.zeros(3, np.float32), np.ones(3, np.float32))
    return st


def same(a, b):
    # (a pull puts the boundary into cell order; its ids are unique)
    oa, ob = np.argsort(a.boundary_id), np.argsort(b.boundary_id)
    np.testing.assert_array_equal(a.fluid_id, b.fluid_id)
    np.testing.assert_array_equal(a.boundary_id[oa], b.boundary_id[ob])
    np.testing.assert_array_equal(a.rigid_id, b.rigid_id)
    np.testing.assert_array_equal(a.rigid_body, b.rigid_body)
    for k in a.boundary:
        np.testing.assert_array_equal(a.boundary[k][oa].view(np.uint32), b.boundary[k][ob].view(np.uint32), err_msg=k)
    for ga, gb in ((a.fluid, b.fluid), (a.rigid, b.rigid), (a.body, b.body)):
        for k in ga:
            np.testing.assert_array_equal(ga[k].view(np.uint32), gb[k].view(np.uint32), err_msg=k)


# 18 words a fluid particle: 116508 of them fill one 8 MiB buffer, 262145 take three
@pytest.mark.parametrize("n", [(1, 0, 0, 0), (1, 1, 1, 1), (255, 1023, 63, 2), (1024, 1025, 1024, 3), (4099, 0, 2049, 1),
                               (116507, 0, 0, 0), (116509, 7, 0, 0), (262145, 100003, 5001, 5)])
def test_round_trip(n):
    print(f"case: round trip {n}", flush=True)
    st = random_state(n, sum(n))
    g = HipBackend()
    g.set_params(scenes.make_params(0.01))
    g.pull(st)
    same(g.push(), st)
    # a second scene, smaller or larger, through the buffers that the first one left
    st2 = random_state((n[0] // 3 + 1, n[1] * 2, n[2], n[3]), 7)
    g.pull(st2)
    same(g.push(), st2)


def test_several_scenes():
    sizes = [(300, 17, 9, 1), (1, 0, 0, 0), (70000, 3000, 0, 0), (2047, 0, 333, 2)]
    states = [random_state(n, 100 + i) for i, n in enumerate(sizes)]
    b = HipBatch()
    ids = b.update(add=[(scenes.make_params(0.01), s) for s in states])
    for i, s in zip(ids, states):
        same(b.push(i), s)
    more = random_state((513, 31, 12, 1), 200)
    ids2 = b.update(remove=[ids[0]], add=[(scenes.make_params(0.01), more)])
    for i, s in zip(ids[1:] + ids2, states[1:] + [more]):
        same(b.push(i), s)


def test_missing_fields():
    n = (1500, 700, 300, 2)
    st = random_state(n, 5)
    p = scenes.make_params(0.01)
    g = HipBackend()
    g.set_params(p)
    g.set_domain(*st.domain)
    v = st.view()
    null_f, null_u64 = ctypes.POINTER(ctypes.c_float)(), ctypes.POINTER(ctypes.c_uint64)()
    for i, k in enumerate(_capi.F_FIELDS):
        if k not in ("x", "y", "z"):
            v.fluid[i] = null_f
    for i, k in enumerate(_capi.B_FIELDS):
        if k not in ("x", "y", "z"):
            v.boundary[i] = null_f
    for i in range(len(_capi.R_FIELDS)):
        v.rigid[i] = null_f
    for i in range(len(_capi.RB_FIELDS)):
        v.body[i] = null_f
    v.fluid_id = v.boundary_id = v.rigid_id = null_u64
    g._check(g.lib.tsp_pull(g.h, ctypes.byref(v)), "tsp_pull")
    g.n = n
    out = g.push()
    for k, f in out.fluid.items():
        np.testing.assert_array_equal(f, st.fluid[k] if k in "xyz" else 0)
    mass = np.float32(np.float32(p.rest_density) * np.float32(p.particle_size) * np.float32(p.particle_size)
                      * np.float32(p.particle_size))
    want = {"psi": mass, "vol": mass / np.float32(p.rest_density)}
    back = out.boundary_id.astype(np.int64)
    for k, f in out.boundary.items():
        np.testing.assert_array_equal(f, st.boundary[k][back] if k in "xyz" else want[k])
    for f in out.rigid.values():
        np.testing.assert_array_equal(f, 0)
    for k, f in out.body.items():
        np.testing.assert_array_equal(f, 1 if k.lower() in ("a00", "a11", "a22") else 0, err_msg=k)
    for f in (out.fluid_id, np.sort(out.boundary_id), out.rigid_id):
        np.testing.assert_array_equal(f, np.arange(f.size))
