"""Fluid sweeps at all strip widths (16, 8 and 4 lines for fluids of 128, 256 and
512 cells), with cells whose divisions leave the fast path beside ordinary ones.

A periodic pattern of 64^3 cells repeated through a fluid evolves into the
repeated result of the pattern, bit for bit, so the restatement evolves the
pattern alone (bars of the sweep test in test_fluid.py: 1e-6 relative, 1e-7
absolute)."""
import numpy as np
import pytest

import oracle_lib as ol
from cube_nufluid_amd.checkpoint import neu_ncb
from cube_nufluid_amd.params import BoxConfig
from test_gpu_fluid_paths import G, mixed_state

M = 64


@pytest.mark.gpu
def test_gpu_sweeps_at_all_strip_widths():
    from cube_nufluid_amd.driver import Cube
    cfg = BoxConfig(nc=256, nnt=1, ncb=6, box=100.0, np_nc=1)
    cube = Cube.from_ic(cfg, 3, 10.0)
    try:
        cube.nu_init(m_ev=0.1, f_neu=0.0075, z_i_nu=10.0)
        for kind in ("tiny", "patches"):
            start = [mixed_state(M, 90 + n, kind) for n in range(3)]
            for n in range(3):
                k = cube.nu_info(n)["nc"] // M
                cube.nu_set(n, np.tile(start[n], (1, k, k, k)))
            cube.dt_neu = np.float32(1000)
            cube.fluid_evolve(0.1, 1, 0.5)
            dt_all = 1000.0
            for n in range(3):
                info = cube.nu_info(n)
                k = info["nc"] // M
                ref, dt_all = ol.fluid_evolve(start[n], neu_ncb(info["dx"]), G, 0.1, info["dx"], 1, dt_all)
                got = cube.nu_get(n).reshape(5, k, M, k, M, k, M)
                first = got[:, 0, :, 0, :, 0, :]
                print(kind, "nc", info["nc"], "max abs diff", float(np.abs(first - ref).max()), flush=True)
                np.testing.assert_allclose(first, ref, rtol=1e-6, atol=1e-7)
                assert (got == first[:, None, :, None, :, None, :]).all()
            assert abs(float(cube.dt_neu) / dt_all - 1) < 1e-6
    finally:
        cube.close()
