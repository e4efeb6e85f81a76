"""Initial conditions' binning where its paths change, against the host twin: one
particle a cell, runs of several, a box so clustered that a workgroup's 256
cells hold more particles (over 4096 here) than are sorted in LDS.

The GPU's transforms run in FP32, the host's in FP64: 18 levels of butterflies
at 6e-8 each leave some 1e-6 of the largest displacement or velocity, so a few
in-cell codes in a hundred land one unit apart and a cell's mean velocity is
within 1e-5 of the largest velocity where the same particles are in the cell."""
import numpy as np
import pytest

from cube_nufluid_amd.params import BoxConfig
from cube_nufluid_amd.ic import zeldovich_ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_nc,box,z", [(1, 100.0, 9.0), (2, 100.0, 9.0), (2, 50.0, 0.5)],
                         ids=["one_a_cell", "eight_a_cell", "clustered"])
def test_binning_matches_host(np_nc, box, z):
    from cube_nufluid_amd.driver import Cube
    cfg = BoxConfig(nc=32, nnt=2, ncb=6, np_nc=np_nc, box=box)
    h = zeldovich_ic(cfg, seed=77, z=z)
    most = int(h.rhoc.reshape(-1, 256).sum(1).max())
    print("np_nc", np_nc, "box", box, "z", z, "fullest 256 cells", most, flush=True)
    assert (most > 4096) == (z < 1)
    cube = Cube.from_ic(cfg, seed=77, z=z)
    g = cube.download()
    cube.close()
    assert g.sim.nplocal == h.sim.nplocal and abs(g.sim.sigma_vi - h.sim.sigma_vi) <= 1e-4 * h.sim.sigma_vi
    assert abs(g.sim.vz_max - h.sim.vz_max) <= 1e-5 * h.sim.vz_max
    nc3 = cfg.nc ** 3
    cg, ch = np.repeat(np.arange(nc3), g.rhoc.reshape(-1)), np.repeat(np.arange(nc3), h.rhoc.reshape(-1))
    assert np.all((np.diff(cg) > 0) | (np.diff(g.pid) > 0))
    og, oh = np.argsort(g.pid), np.argsort(h.pid)
    np.testing.assert_array_equal(g.pid[og], h.pid[oh])
    same = cg[og] == ch[oh]
    assert np.mean(same) > 0.999
    du = np.abs(g.xp[og].view(np.uint16).astype(np.int64) - h.xp[oh].view(np.uint16).astype(np.int64))
    assert np.max(du[same]) <= 1 and np.mean(du[same] == 0) > 0.97
    moved = np.zeros(nc3, dtype=bool)
    moved[cg[og][~same]] = True
    moved[ch[oh][~same]] = True
    dv = np.abs(g.vfield.reshape(nc3, 3) - h.vfield.reshape(nc3, 3))[~moved]
    assert np.max(dv) <= 1e-5 * np.max(np.abs(h.vfield))
