"""Fluid sweeps at the far end of the floats: momenta whose squares overflow,
cells with next to no mass, infinite momenta and pressures near the largest
float, a few of them among ordinary cells.

Where a quotient overflows the restatement's plain division gives an infinity,
and an infinite sound speed a zero time step, so the sweep has to give the same
infinities and NaNs in the same cells and the same step.  Finite values keep the
bars of the sweep test in test_fluid.py (1e-6 relative, 1e-7 absolute) where no
NaN reaches them: the limiter reads a NaN's sign, which no standard fixes and
host and GPU set differently, and the three sweeps carry it two cells along each
axis."""
import numpy as np
import pytest

import oracle_lib as ol
from cube_nufluid_amd.checkpoint import neu_ncb
from cube_nufluid_amd.params import BoxConfig
from test_gpu_fluid_paths import G, mixed_state


def extreme_state(nc, seed, kind):
    f = mixed_state(nc, seed, "full")
    rng = np.random.default_rng(seed + 1000)
    hot = rng.permutation(nc ** 3).reshape(nc, nc, nc) < 8
    if kind == "momenta":
        f[1:4, hot] = 10.0 ** rng.uniform(18, 24, (3, 8)) * rng.choice([-1, 1], (3, 8))
    elif kind == "thin":
        f[0, hot] = 10.0 ** rng.uniform(-14, -9, 8)
        f[1:4, hot] = 10.0 ** rng.uniform(0, 26, (3, 8))
    elif kind == "infinite":
        f[1:4, hot] = np.inf
    else:
        f[4, hot] = 10.0 ** rng.uniform(20, 38, 8)
    return f


def clear_of_nan(ref):
    near = ~np.isfinite(ref).all(0)
    for ax in range(3):
        near = np.any([np.roll(near, k, ax) for k in range(-2, 3)], 0)
    return ~near


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["momenta", "thin", "infinite", "pressure"])
def test_gpu_sweeps_overflow(kind):
    from cube_nufluid_amd.driver import Cube
    from cube_nufluid_amd.ic import zeldovich_ic
    cfg = BoxConfig(nc=16, nnt=1, ncb=6, box=100.0)
    ic = BoxConfig(nc=16, nnt=1, ncb=6, box=100.0, np_nc=1)
    cube = Cube(cfg, zeldovich_ic(ic, seed=3, z=10.0))
    cube.nu_init(m_ev=0.1, f_neu=0.0075, z_i_nu=10.0)
    try:
        start = []
        for n in range(3):
            start.append(extreme_state(cube.nu_info(n)["nc"], 70 + n, kind))
            cube.nu_set(n, start[n])
        cube.dt_neu = np.float32(1000)
        cube.fluid_evolve(0.1, 1, 0.5)
        dt_all = 1000.0
        for n in range(3):
            info = cube.nu_info(n)
            with np.errstate(all="ignore"):
                ref, dt_all = ol.fluid_evolve(start[n], neu_ncb(info["dx"]), G, 0.1, info["dx"], 1, dt_all)
            got = cube.nu_get(n)
            print(kind, info["nc"], "infinities", int(np.isinf(ref).sum()), "NaNs", int(np.isnan(ref).sum()), flush=True)
            np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
            np.testing.assert_array_equal(got == np.inf, ref == np.inf)
            np.testing.assert_array_equal(got == -np.inf, ref == -np.inf)
            clear = clear_of_nan(ref)
            np.testing.assert_allclose(got[:, clear], ref[:, clear], rtol=1e-6, atol=1e-7)
        assert abs(float(cube.dt_neu) - dt_all) <= 1e-6 * dt_all
    finally:
        cube.close()
