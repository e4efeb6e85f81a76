"""The fluids take their five fields, and gravity accumulators (four doubles a
cell) only for the third: the gathers of the other two update the cells
themselves."""
import pytest

from cube_nufluid_amd.params import BoxConfig
from test_footprint import free_memory


@pytest.mark.gpu
@pytest.mark.parametrize("nc", [64, 128])
def test_gpu_fluid_allocations(nc):
    from cube_nufluid_amd.driver import Cube
    cfg = BoxConfig(nc=nc, nnt=1, ncb=6, box=100.0, np_nc=1)
    cube = Cube.from_ic(cfg, 3, 10.0)
    try:
        free = free_memory(cube.lib)
        cube.nu_init(m_ev=0.1, f_neu=0.0075, z_i_nu=10.0)
        used = free - free_memory(cube.lib)
        cells = [cube.nu_info(n)["nc"] ** 3 for n in range(3)]
        need = 20 * sum(cells) + 32 * cells[2]
        print("nc", nc, "taken", used, "fields and accumulators", need, flush=True)
        assert used <= need + 16e6  # four allocations, each rounded up by the runtime
    finally:
        cube.close()
