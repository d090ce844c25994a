"""The statistics kernels at the sizes where they can go wrong, against numpy on the pushed state and the decoded
lists: no particle, one block that is not full, several, counts beyond the bins kept in LDS (a block squeezed
into one support radius: 600 and more neighbors), all particles in one bin (a single particle repeated), and a
scene with rigid particles.
"""
import numpy as np
import pytest

from turbospharticles_amd import _capi, scenes
from turbospharticles_amd.backend import HipBackend

from helpers import cube_scene, dam_break

pytestmark = pytest.mark.gpu

H = 0.01


def squeezed():
    st = dam_break(10, H, counts=(10, 8, 8), tank=(0.3, 0.2, 0.2))
    for f in "xyz":
        st.fluid[f][:] = np.float32(0.1) + (st.fluid[f] - np.float32(0.1)) * np.float32(0.12)
    return st


CASES = {
    "none": lambda: _capi.HostState(0, 0, 0, 0),
    "one": lambda: dam_break(1, H, counts=(1, 1, 1), tank=(0.1, 0.1, 0.1)),
    "315": lambda: dam_break(5, H, counts=(5, 7, 9), tank=(0.2, 0.2, 0.2)),
    "squeezed": squeezed,
    "cube": lambda: cube_scene(center=(0.15, 0.035, 0.15)),
    "70,000": lambda: dam_break(40, H, counts=(40, 35, 50), tank=(1.0, 0.5, 0.6)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_statistics_match_numpy(name):
    print(f"case: {name}", flush=True)
    st = CASES[name]()
    p = scenes.make_params(H)
    rng = np.random.default_rng(3)
    for f in ("vx", "vy", "vz"):
        st.fluid[f][:] = rng.normal(0.0, 0.5, st.n[0]).astype(np.float32)
    st.fluid["density"][:] = rng.normal(1000.0, 5.0, st.n[0]).astype(np.float32)
    g = HipBackend(0)
    g.set_params(p)
    g.pull(st)
    g.neighbor_search()
    s = g.statistics()
    out = g.push()
    n = st.n
    assert (s.n_fluid, s.n_boundary, s.n_rigid) == n[:3]
    for rel in range(6):
        c = np.sort(g.neighbors(rel)[0].astype(np.int64)) if n[0 if rel < 3 else 2] else np.zeros(0, np.int64)
        if c.size == 0:
            assert (s.nbr_min[rel], s.nbr_max[rel], s.nbr_p99[rel], s.nbr_avg[rel]) == (0, 0, 0, 0.0), rel
            continue
        assert (s.nbr_min[rel], s.nbr_max[rel]) == (c[0], c[-1]), rel
        assert s.nbr_p99[rel] == c[(99 * (c.size - 1)) // 100], rel
        assert s.nbr_avg[rel] == c.sum() / c.size, rel   # whole numbers below 2^53: one division on either side
    if name == "squeezed":
        assert s.nbr_max[0] >= 600
    if n[0]:
        e = (out.fluid["density"] / np.float32(p.rest_density) - np.float32(1.0)).astype(np.float64)
        # float32 terms summed in float64 in any order: n 2^-53 relative to the sum of magnitudes
        tol = 2.0 ** -50 * n[0]
        for got, term in zip(s.dens_rel_err_avg, (e, np.maximum(e, 0.0), np.abs(e))):
            assert abs(got - term.mean()) <= tol * np.abs(e).mean()
        v = [out.fluid[f].astype(np.float64) for f in ("vx", "vy", "vz")]
        m = np.sqrt(v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
        # |v| in float32: three roundings of the square, one of the root
        for got, want in ((s.vel_avg, m.mean()), (s.vel_min, m.min()), (s.vel_max, m.max())):
            assert abs(got - want) <= 4 * 2.0 ** -24 * want + 1e-30
    g.close()
