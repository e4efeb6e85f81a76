"""Branches of the GPU halo finder that the catalogue tests do not reach: a
halo wider than the short offset table, search lists on both sides of the LDS
sort's size, and more halos than one chunk of the running sums.

Members, order and the halo_pid stream are whole numbers and equal the
restatement's; float fields carry FP32 rounding of per-halo sums (bars of
test_halo.py's compare)."""
import numpy as np
import pytest

import oracle_lib as ol
from cube_nufluid_amd.halo import HaloParams
from cube_nufluid_amd.params import BoxConfig
from test_halo import clumps_state, compare, gpu_catalog


def broad_state(cfg, seed):
    """A ball 9 coarse cells in radius around a dense core."""
    from cube_nufluid_amd.ic import encode_particles
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(40000, 3))
    d *= 9.0 * rng.uniform(size=(40000, 1)) ** (1 / 3) / np.linalg.norm(d, axis=1)[:, None]
    core = rng.normal(0, 0.15, size=(3000, 3))
    pos = np.concatenate([np.array([16.2, 15.9, 16.4]) + d, np.array([16.2, 15.9, 16.4]) + core,
                          rng.uniform(0, cfg.nc, size=(4000, 3))])
    vel = rng.normal(0, 0.5, size=pos.shape)
    return encode_particles(cfg, pos, vel, np.arange(1, len(pos) + 1, dtype=np.int32), np.float32(1.0))


def case(name):
    if name == "broad":
        cfg = BoxConfig(nc=32, nnt=1, ncb=6, box=100.0)
        # 34000 particles on the mesh make a peak: only the walk past 32 cells
        # counts that many.  Its search list (20 cells) stays above the
        # overdensity, so it is processed without becoming a halo.
        hp = HaloParams(den_odc=5.0, den_peak_cutoff=9000.0, nc_halo_max=60, min_halo_particles=68000)
        return cfg, broad_state(cfg, 3), hp.for_box(cfg)
    if name == "many":
        cfg = BoxConfig(nc=64, nnt=2, ncb=6, box=200.0)
        rng = np.random.default_rng(5)
        grid = (np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * (cfg.nc / 6)
        specs = [(c + rng.uniform(-2, 2, 3), int(rng.integers(300, 500)), 0.12) for c in grid]
        return cfg, clumps_state(cfg, specs, 200000, seed=6), HaloParams(min_halo_particles=20, nc_halo_max=12).for_box(cfg)
    cfg = BoxConfig(nc=16, nnt=2, ncb=6, box=50.0)
    specs = [((4.1, 4.3, 3.8), 4000, 0.3), ((12.2, 11.9, 4.4), 4300, 0.3), ((4.0, 12.0, 12.3), 9000, 0.3)]
    return cfg, clumps_state(cfg, specs, 15000, seed=9), HaloParams(nc_halo_max=40).for_box(cfg)


@pytest.mark.gpu
@pytest.mark.parametrize("name,peaks,least", [("broad", 1, 0), ("many", 129, 129), ("list_sizes", 3, 3)])
def test_gpu_halofind_paths(name, peaks, least):
    cfg, st, hp = case(name)
    halos, words, hid, counts = ol.halofind(cfg, st, hp, nhid=st.sim.nplocal)
    print(name, "oracle: %d halos, %d peaks processed" % (len(halos), counts[3]), flush=True)
    cat = gpu_catalog(cfg, st, hp, nhid=st.sim.nplocal)
    assert cat.nprocessed == counts[3] >= peaks
    assert cat.nhalo == len(halos) >= least
    if least:
        compare(cat, halos, words, hid, cfg.nf)
