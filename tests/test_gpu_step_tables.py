"""The decode tables and the scalars that a step leaves on the device for the
next one: a drift that fails between two steps, a kick repeated without a drift
and a table asked for in between leave what follows unchanged, bit for bit,
for both velocity widths."""
import numpy as np
import pytest

from cube_nufluid_amd.params import BoxConfig

pytestmark = pytest.mark.gpu


def fields(cube):
    st = cube.download()
    return [np.array(getattr(st, f)) for f in ("xp", "vp", "pid", "rhoc", "vfield")]


def run(izipv, upset):
    from cube_nufluid_amd.driver import Cube
    cfg = BoxConfig(nc=16, nnt=2, ncb=6, izipv=izipv, box=50.0, pp_on=True)
    cube = Cube.from_ic(cfg, 5, 9.0)
    cube.a_mid = np.float32(0.1)
    outs = []
    for step in range(4):
        if upset and step == 2:
            # past ncb coarse cells in one drift, refused after its launches
            cube.dt_old = cube.dt = np.float32(40 / cube.sim.vz_max)  # 10 coarse cells
            with pytest.raises(RuntimeError):
                cube.update_x()
        if upset and step == 3:
            cube.probe_pm_forces()
            cube.probe_pp_forces()
        cube.dt_old = cube.dt = np.float32(0.02 * (step + 1))
        g = cube.update_x()
        p = cube.particle_mesh()
        p = cube.particle_mesh()  # a second kick, old and new sigma now equal
        outs.append((float(g.sigma_vi_new), float(p.f2_max_coarse), float(p.f2_max_fine), tuple(p.vmax), g.npcheck))
    f = fields(cube)
    cube.close()
    return outs, f


@pytest.mark.parametrize("izipv", [1, 2])
def test_tables_between_steps(izipv):
    print("izipv", izipv, flush=True)
    a, fa = run(izipv, False)
    b, fb = run(izipv, True)
    assert a == b
    assert all(o[1] > 0 and o[2] > 0 and min(o[3]) > 0 for o in a)
    for x, y in zip(fa, fb):
        np.testing.assert_array_equal(x, y)
