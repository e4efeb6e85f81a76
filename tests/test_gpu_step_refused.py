"""A step refused because a particle moves past the buffer, in each step mode:
in modes 1 and 2 PP and both kicks have already run on the refused drift's
result, with the decode tables of its sigma.  The box keeps its state, and the
steps that follow give the bits of a run without the refusals."""
import ctypes

import numpy as np
import pytest

from cube_nufluid_amd import _lib
from cube_nufluid_amd.params import BoxConfig

STEPS = 6


def run(izipv, mode, refuse_at):
    from cube_nufluid_amd.driver import Cube
    cfg = BoxConfig(nc=16, nnt=2, ncb=6, izipv=izipv, box=50.0, pp_on=True)
    cube = Cube.from_ic(cfg, 5, 9.0)
    lib, clk = cube.lib, _lib.CubeClock()
    try:
        _lib.check(lib, cube.h, lib.cube_set_step_mode(cube.h, mode))
        z = np.array([9.0, 0.0], dtype=np.float32)
        assert lib.cube_clock_init(ctypes.byref(clk), _lib.ptr(z), 2) == 0
        clocks = []
        for step in range(STEPS):
            for _ in range(refuse_at.count(step)):
                far = _lib.CubeClock.from_buffer_copy(clk)
                # half of the step before is 10 coarse cells long: past the
                # buffer of 6, below the 15 that are refused before the launches
                far.dt = 80.0 / cube.download().sim.vz_max
                rc = lib.cube_step(cube.h, ctypes.byref(far))
                err = ctypes.create_string_buffer(256)
                lib.cube_last_error(cube.h, err, 256)
                assert rc != 0 and b"coarse cells in one drift" in err.value
            _lib.check(lib, cube.h, lib.cube_step(cube.h, ctypes.byref(clk)))
            clocks.append((clk.a, clk.dt, clk.a_mid))
        st = cube.download()
        return clocks, [np.array(getattr(st, f)) for f in ("xp", "vp", "pid", "rhoc", "vfield")]
    finally:
        cube.close()


@pytest.mark.gpu
@pytest.mark.parametrize("izipv", [1, 2])
def test_refused_steps_leave_no_trace(izipv):
    want = run(izipv, 0, [])
    assert len(set(want[0])) == STEPS
    for mode in (0, 1, 2):
        for refuse_at in ([0], [2, 2], [1, 3, 4]):
            print("izipv", izipv, "mode", mode, "refused before steps", refuse_at, flush=True)
            got = run(izipv, mode, refuse_at)
            assert got[0] == want[0]
            for x, y in zip(got[1], want[1]):
                np.testing.assert_array_equal(x, y)
