"""Fluid sweeps where their divisions leave the fast path: cells at rest,
momenta down to the denormals, empty differences, beside ordinary cells, at
the strip widths of small and larger fluids.

The sweep evaluates the restatement's float expressions one by one with
correctly rounded divisions, so it differs at most where the host compiler
orders a sum differently: the bars of the sweep test in test_fluid.py (1e-6
relative, 1e-7 absolute)."""
import numpy as np
import pytest

import oracle_lib as ol
from cube_nufluid_amd.checkpoint import neu_ncb
from cube_nufluid_amd.params import BoxConfig

G = np.float32(5.0 / 3.0)


def mixed_state(nc, seed, kind):
    rng = np.random.default_rng(seed)
    f = np.empty((5, nc, nc, nc), dtype=np.float32)
    f[0] = 1 + 0.1 * rng.standard_normal((nc, nc, nc))
    f[1:4] = 0.05 * rng.standard_normal((3, nc, nc, nc))
    if kind == "rest":
        f[0], f[1:4] = 1.0, 0.0
    elif kind == "patches":
        still = rng.random((nc, nc, nc)) < 0.5
        f[1:4, still] = 0.0
        f[1, ~still] = -0.0
    elif kind == "tiny":
        f[1:4] = (f[1:4] * 10.0 ** rng.uniform(-40, 0, f[1:4].shape)).astype(np.float32)
    f[4] = f[0] * 0.3 + (f[1:4].astype(np.float64) ** 2).sum(0) / (2 * f[0])
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("nc,kind", [(16, "rest"), (16, "patches"), (16, "tiny"), (16, "full"), (64, "tiny"), (64, "patches")])
def test_gpu_sweeps_off_the_fast_division(nc, kind):
    from cube_nufluid_amd.driver import Cube
    from cube_nufluid_amd.ic import zeldovich_ic
    cfg = BoxConfig(nc=nc, nnt=1, ncb=6, box=100.0)
    ic = BoxConfig(nc=nc, nnt=1, ncb=6, box=100.0, np_nc=1)
    cube = Cube(cfg, zeldovich_ic(ic, seed=3, z=10.0))
    cube.nu_init(m_ev=0.1, f_neu=0.0075, z_i_nu=10.0)
    try:
        for n in range(3):
            info = cube.nu_info(n)
            cube.nu_set(n, mixed_state(info["nc"], 50 + n, kind))
        start = [cube.nu_get(n) for n in range(3)]
        cube.dt_neu = np.float32(1000)
        cube.fluid_evolve(0.1, 1, 0.5)
        dt_all = 1000.0
        for n in range(3):
            info = cube.nu_info(n)
            ref, dt_all = ol.fluid_evolve(start[n], neu_ncb(info["dx"]), G, 0.1, info["dx"], 1, dt_all)
            got = cube.nu_get(n)
            print("nc", info["nc"], kind, "max abs diff", float(np.abs(got - ref).max()), flush=True)
            np.testing.assert_allclose(got, ref, rtol=1e-6, atol=1e-7)
        assert abs(float(cube.dt_neu) / dt_all - 1) < 1e-6
    finally:
        cube.close()
