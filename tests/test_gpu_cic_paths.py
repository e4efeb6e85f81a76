"""CIC mass assignment at the sizes where its paths change, against the oracle:
cells mostly empty, several particles a cell, more particles in a block than
one batch, particles too heavy for the fast rounding, half- and full-width
coarse blocks, both position widths.

The GPU's node sums are exact in 2^-40 units.  The oracle adds n float weights
one after the other, each addition off by at most 2^-24 of the running sum, so
a node of value v differs by at most (n + 2) 2^-24 v + n 2^-40, n being at most
eight times the fullest cell.  The coarse mesh is seen through its forces, to
the 1e-5 relative RMS of the force parity bar."""
import numpy as np
import pytest

from cube_nufluid_amd.params import BoxConfig

pytestmark = pytest.mark.gpu

CASES = [
    ("sparse", 16, 2000, 0, 2),
    ("sparse_x1", 16, 2000, 0, 1),
    ("heavy", 16, 60, 0, 2),
    ("heavy_x1", 16, 60, 0, 1),
    ("dense_batches", 16, 40000, 0, 2),
    ("dense_batches_x1", 16, 40000, 0, 1),
    ("clump", 16, 4000, 400, 2),
    ("wide_sparse", 64, 100000, 0, 2),
    ("wide_sparse_batches", 64, 600000, 0, 2),
    ("wide_dense_batches", 64, 1200000, 0, 2),
    ("wide_dense_x1", 64, 1200000, 0, 1),
]


@pytest.mark.parametrize("name,nc,n,clump,izipx", CASES, ids=[c[0] for c in CASES])
def test_cic_paths(name, nc, n, clump, izipx):
    from cube_nufluid_amd.driver import Cube
    from cube_nufluid_amd.ic import encode_particles
    from oracle_lib import Oracle
    cfg = BoxConfig(nc=nc, nnt=2, ncb=6, izipx=izipx, box=50.0)
    rng = np.random.default_rng(n + izipx)
    pos = rng.uniform(0, nc, size=(n, 3))
    if clump:
        pos = np.concatenate([pos, rng.normal(nc / 2 + 0.3, 0.2, size=(clump, 3))])
    st = encode_particles(cfg, pos, rng.normal(0, 0.5, size=pos.shape), np.arange(1, len(pos) + 1, dtype=np.int32), np.float32(0.5))
    print("case", name, "fullest cell", int(st.rhoc.max()), flush=True)
    cube, orc = Cube(cfg, st), Oracle(cfg)
    orc.set_state(st)
    g, o = cube.probe_density().astype(np.float64), orc.density().astype(np.float64)
    m = 8 * int(st.rhoc.max())
    assert np.all(np.abs(g - o) <= (m + 2) * 2.0 ** -24 * o + m * 2.0 ** -40)
    assert abs(g.sum() - cfg.nf ** 3) <= 1e-6 * cfg.nf ** 3
    fc, oc = cube.probe_pm_forces()[1], orc.pm_forces()[1]
    assert np.sqrt(np.mean((fc - oc) ** 2)) < 1e-5 * np.sqrt(np.mean(oc ** 2))
    cube.close()
