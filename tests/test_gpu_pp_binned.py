"""The binned PP kernel and the dense-block pair sums at the sizes where they
can go wrong, against the oracle: every reach, both position widths, cells
without particles, regions larger than the owner table whose window holds few
candidates, runs longer than the whole-number sums allow.

Forces are FP32 pairs summed in double or 2^-32 units against the oracle's
FP64 pairs stored as FP32: each pair carries a few FP32 roundings (some 6e-8
each), and opposite pairs cancel by up to a factor of ten in a clump, so the
relative RMS stays below the 1e-5 of the force parity bar."""
import numpy as np
import pytest

from cube_nufluid_amd.params import BoxConfig

pytestmark = pytest.mark.gpu


def state(cfg, parts, seed):
    """parts: (count, centre in coarse cells or None for uniform, sigma)"""
    from cube_nufluid_amd.ic import encode_particles
    rng = np.random.default_rng(seed)
    pos = np.concatenate([rng.uniform(0, cfg.nc, size=(n, 3)) if c is None else rng.normal(c, s, size=(n, 3))
                          for n, c, s in parts])
    vel = rng.normal(0, 0.5, size=pos.shape)
    return encode_particles(cfg, pos, vel, np.arange(1, len(pos) + 1, dtype=np.int32), np.float32(0.5))


CASES = [
    # sparse: most fine cells and many coarse cells empty
    *[("sparse_r%d_x%d" % (r, x), dict(pp_range=r, izipx=x), [(3000, None, 0)]) for r in (1, 2, 3, 4) for x in (1, 2)],
    # a few hundred candidates a block, runs of several particles
    *[("clump_r%d" % r, dict(pp_range=r), [(900, 7.9, 0.5), (9000, None, 0)]) for r in (1, 2, 3, 4)],
    # a tight clump in the middle of one coarse cell: neighbouring blocks see
    # more region particles than the owner table holds, but not in their window
    ("far_from_window_r1", dict(pp_range=1), [(5000, 4.5, 0.02), (4000, None, 0)]),
    ("far_from_window_r3", dict(pp_range=3), [(2500, 4.5, 0.02), (2000, None, 0)]),
    # dense blocks; a softening for which only the 64-bit sums are exact
    ("dense_small_softening", dict(pp_range=1, rsoft=0.002), [(4000, 8.1, 0.4), (4000, None, 0)]),
    ("dense_r2", dict(pp_range=2), [(4000, 8.1, 0.4), (4000, None, 0)]),
]


@pytest.mark.parametrize("name,kw,parts", CASES, ids=[c[0] for c in CASES])
def test_pp_binned(name, kw, parts):
    from cube_nufluid_amd.driver import Cube
    from oracle_lib import Oracle
    cfg = BoxConfig(nc=16, nnt=2, ncb=6, box=50.0, pp_on=True, **kw)
    st = state(cfg, parts, seed=len(name))
    print("case", name, st.sim.nplocal, "largest cell", int(st.rhoc.max()), flush=True)
    cube = Cube(cfg, st)
    orc = Oracle(cfg)
    orc.set_state(st)
    gp = cube.probe_pp_forces()
    r = orc.pp(1.0, 1.0, forces=True)
    op = r["f_pp"].astype(np.float64)
    err = float(np.sqrt(np.mean((gp - op) ** 2)) / np.sqrt(np.mean(op ** 2)))
    print("relative RMS", err, flush=True)
    cube.a_mid, cube.dt = np.float32(0.2), np.float32(0.05)
    o = cube.ext_pp_force()
    cube.close()
    assert err < 1e-5
    assert o.npairs == r["npairs"] and o.itest1 == st.sim.nplocal
