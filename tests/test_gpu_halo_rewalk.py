"""The mesh walk repeated with the full offset table, which one peak that reaches
past the short one (32 fine cells) asks for: halos of the same call, and the
mesh mass itself, bounded on both sides by the particle count that a peak needs.

Counts, members and the halo_pid stream are whole numbers and equal the
restatement's; float fields keep the bars of test_halo.py's compare."""
import numpy as np
import pytest

import oracle_lib as ol
from cube_nufluid_amd.halo import HaloParams
from cube_nufluid_amd.params import BoxConfig
from test_halo import compare, gpu_catalog

CENTRE = np.array([16.2, 15.9, 16.4])


def state(cfg, specs, seed):
    """A ball 9 coarse cells in radius around a dense core, and clumps."""
    from cube_nufluid_amd.ic import encode_particles
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(40000, 3))
    d *= 9.0 * rng.uniform(size=(40000, 1)) ** (1 / 3) / np.linalg.norm(d, axis=1)[:, None]
    parts = [CENTRE + d, CENTRE + rng.normal(0, 0.15, size=(3000, 3)), rng.uniform(0, cfg.nc, size=(4000, 3))]
    parts += [np.asarray(c) + rng.normal(0, s, size=(n, 3)) for c, n, s in specs]
    pos = np.concatenate(parts) % cfg.nc
    vel = rng.normal(0, 0.5, size=pos.shape)
    return encode_particles(cfg, pos, vel, np.arange(1, len(pos) + 1, dtype=np.int32), np.float32(1.0))


def walk_mass(cfg, st, hp):
    """(mesh mass, number of offsets taken) of the walk from the densest node."""
    rho = ol.halo_density(cfg, st, hp)
    k, j, i = np.unravel_index(np.argmax(rho), rho.shape)
    t = ol.halo_offset_table(hp.nc_halo_max)
    m = np.cumsum(rho[(k + t[:, 2]) % cfg.nf, (j + t[:, 1]) % cfg.nf, (i + t[:, 0]) % cfg.nf].astype(np.float64))
    n = np.arange(1, len(t) + 1)
    shell = np.append(t[1:, 3] != t[:-1, 3], True)
    at = int(np.argmax(shell & (n >= 19) & (m / n < hp.den_odc)))
    return m[at], at + 1


@pytest.mark.gpu
@pytest.mark.parametrize("nnt", [1, 2])
def test_gpu_halos_beside_a_long_walk(nnt):
    cfg = BoxConfig(nc=32, nnt=nnt, ncb=6, box=100.0)
    specs = [((0.3, 0.1, 0.8), 700, 0.12), ((0.9, 16.2, 1.0), 500, 0.1), ((15.4, 0.2, 0.9), 900, 0.15),
             ((1.0, 0.3, 16.6), 400, 0.1), ((16.1, 15.3, 0.8), 600, 0.12), ((0.2, 16.4, 15.5), 800, 0.12)]
    st = state(cfg, specs, 3)
    hp = HaloParams(den_odc=5.0, den_peak_cutoff=1500.0, nc_halo_max=60, min_halo_particles=100).for_box(cfg)
    assert nnt > 1 or walk_mass(cfg, st, hp)[1] > len(ol.halo_offset_table(32))
    halos, words, hid, counts = ol.halofind(cfg, st, hp, nhid=st.sim.nplocal)
    print("oracle: %d halos, %d peaks processed" % (len(halos), counts[3]), flush=True)
    assert len(halos) >= 5
    cat = gpu_catalog(cfg, st, hp, nhid=st.sim.nplocal)
    assert cat.nprocessed == counts[3]
    compare(cat, halos, words, hid, cfg.nf)


@pytest.mark.gpu
@pytest.mark.parametrize("share,peaks", [(0.995, 1), (1.005, 0)])
def test_gpu_mass_of_a_long_walk(share, peaks):
    cfg = BoxConfig(nc=32, nnt=1, ncb=6, box=100.0)
    st = state(cfg, [], 4)
    hp = HaloParams(den_odc=5.0, den_peak_cutoff=9000.0, nc_halo_max=60, search_ratio=1).for_box(cfg)
    mass, taken = walk_mass(cfg, st, hp)
    assert taken > len(ol.halo_offset_table(32))
    # a peak counts if its mesh mass exceeds half of min_halo_particles
    hp.min_halo_particles = int(round(2 * share * mass / float(st.sim.mass_p_cdm)))
    halos, words, hid, counts = ol.halofind(cfg, st, hp)
    assert counts[3] == peaks and len(halos) == 0
    cat = gpu_catalog(cfg, st, hp)
    print("walk of %d offsets, mass %g: %d peaks processed" % (taken, mass, cat.nprocessed), flush=True)
    assert cat.nprocessed == peaks and cat.nhalo == 0
