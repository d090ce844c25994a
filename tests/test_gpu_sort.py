"""The radix sort's forms at the sizes where they can go wrong: one block (up to 4, 8 and 16 keys per thread),
tiles of 1,024 keys (up to 2^18), tiles of 2,048, with 32-bit and 64-bit keys. Order and keys of a search equal
the oracle's: particles in a shuffled order, many to a cell, some outside the domain; a boundary given in
reverse."""
import numpy as np
import pytest

from turbospharticles_amd import _capi, scenes
from turbospharticles_amd.backend import HipBackend

import oracle_lib as O
from helpers import dam_break

pytestmark = pytest.mark.gpu

H = 0.01
SIZES = [1, 2, 63, 65, 4096, 4097, 8192, 8193, 16384, 16385, 17409, 65536, 262144, 262145, 264193]


def scene(n, wide):
    side = max(8, int(np.ceil(n ** (1.0 / 3.0))))
    full = dam_break(side, H, tank=(side * H * 1.5, side * H * 1.2, side * H * 1.2))
    pick = np.random.default_rng(n).permutation(side ** 3)[:n]
    nB = full.n[1]
    st = _capi.HostState(n, nB, 0, 0)
    st.fluid_id[:] = full.fluid_id[pick]
    st.boundary_id[:] = full.boundary_id[::-1]
    for k in st.fluid:
        st.fluid[k][:] = full.fluid[k][pick]
    for k in st.boundary:
        st.boundary[k][:] = full.boundary[k][::-1]
    lo, hi = (np.array(d, np.float32) for d in full.domain)
    if wide:   # 2,100 cells along x: Morton ids beyond 2^32
        st.fluid["x"][n // 2:] += np.float32(42.0)
        hi[0] += np.float32(42.0)
    st.fluid["y"][::97] += np.float32(3.0)
    st.domain = (lo, hi)
    return st


@pytest.mark.parametrize("n,wide", [(n, False) for n in SIZES] + [(n, True) for n in (4096, 8193, 16384, 16385, 262145)])
def test_order_equals_the_oracle(n, wide):
    print(f"case: {n} keys, wide {wide}", flush=True)
    st = scene(n, wide)
    p = scenes.make_params(H)
    g = HipBackend(0)
    g.set_params(p)
    g.pull(st)
    o = O.Oracle(p, chunk_width=1)
    o.pull(st)
    for _ in range(2):   # once from the given order, once more from the sorted one
        g.neighbor_search()
        o.neighbor_search()
        order, keys, keys_b = g.sort_state()
        ref_order, ref_keys, _, ref_b = o.order()
        assert np.array_equal(order, ref_order)
        assert np.array_equal(keys, ref_keys)
        assert np.array_equal(keys_b, ref_b)
        gs, os = g.push(), o.push()
        assert np.array_equal(gs.fluid_id, os.fluid_id)
        assert np.array_equal(gs.boundary_id, os.boundary_id)
