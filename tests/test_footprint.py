"""What the Zel'dovich generator allocates, and what cube_footprint counts for
it: two plain padded spectra of its ng^3 lattice (ng^2 (ng+2) floats each) and ng
twiddles, beside tables and partial sums of less than 8 MB."""
import ctypes
import threading

import pytest

from cube_nufluid_amd import _lib


@pytest.mark.parametrize("nc,np_nc", [(16, 1), (32, 2), (64, 1), (128, 2), (256, 2), (512, 2)])
def test_generator_meshes_are_counted(nc, np_nc):
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cube_footprint.restype, lib.cube_footprint.argtypes = _lib.SIGNATURES["cube_footprint"]
    p = _lib.CubeParams()
    ng = nc * np_nc
    p.nc, p.nnt, p.ncb, p.izipx, p.izipv, p.np_max, p.precision = nc, 2, 6, 2, 2, ng ** 3, 4
    meshes = 2 * ng * ng * (ng + 2) * 4 + 8 * ng
    got = lib.cube_footprint(ctypes.byref(p), np_nc) - lib.cube_footprint(ctypes.byref(p), 0)
    assert meshes + meshes // 16 <= got <= 1.07 * meshes + 16 * ng  # a sixteenth for the allocator's rounding


@pytest.mark.parametrize("nc,izipx,precision,per_cell,most", [
    (16, 2, 4, 8, (78817541, 79114021)), (16, 1, 8, 1, (84444014, 84740494)),
    (32, 2, 4, 8, (131452873, 133751817)), (32, 1, 8, 1, (168739381, 171038325)),
    (64, 2, 4, 8, (529871057, 547977553)), (64, 1, 8, 1, (796102213, 814208709)),
    (128, 2, 4, 8, (3623690798, 3767415598)), (256, 1, 8, 1, (43497518422, 44642834262)),
    (512, 2, 4, 8, (221405811458, 230550460162)), (512, 1, 8, 1, (343412781114, 352557429818))])
def test_no_box_asks_for_more_than_before(nc, izipx, precision, per_cell, most):
    """`most`: the footprints without and with the generator before the fine
    mesh's spectrum planes were padded.  A memory budget that a caller set by
    them still admits the box."""
    lib = ctypes.CDLL(_lib.LIB_PATH)
    lib.cube_footprint.restype, lib.cube_footprint.argtypes = _lib.SIGNATURES["cube_footprint"]
    p = _lib.CubeParams()
    p.nc, p.nnt, p.ncb, p.izipx, p.izipv, p.np_max, p.precision = nc, 2, 6, izipx, 2, per_cell * nc ** 3, precision
    for ic, m in zip((0, 2), most):
        got = lib.cube_footprint(ctypes.byref(p), ic)
        assert 0.98 * m < got <= m


def free_memory(lib):
    """Free device memory as the library's own HIP runtime reports it."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.gpu
def test_generator_allocates_what_is_counted():
    from cube_nufluid_amd.driver import Cube
    from cube_nufluid_amd.ic import power_table, velocity_factor
    from cube_nufluid_amd.params import BoxConfig
    cfg = BoxConfig(nc=128, nnt=4, ncb=6, box=400.0)
    cube = Cube.from_ic(cfg, 11, 49.0)
    ng = cfg.nc * cfg.np_nc
    lnk, lnp = power_table(cfg, 0.02)
    ip = _lib.ICParams()
    ip.seed, ip.np_nc, ip.nk, ip.a, ip.box = 11, cfg.np_nc, len(lnk), 0.02, cfg.box
    ip.vfac, ip.lnk, ip.lnp, ip.f_cdm = velocity_factor(cfg, 0.02), _lib.ptr(lnk), _lib.ptr(lnp), cfg.f_cdm
    stop, least = threading.Event(), []

    def watch():
        low = free
        while not stop.is_set():
            low = min(low, free_memory(cube.lib))
        least.append(low)

    free = free_memory(cube.lib)
    t = threading.Thread(target=watch)
    t.start()
    try:
        for _ in range(5):
            _lib.check(cube.lib, cube.h, cube.lib.cube_ic_zeldovich(cube.h, ctypes.byref(ip), None))
    finally:
        stop.set()
        t.join()
        cube.close()
    used = free - least[0]
    print("generator's allocations, MB:", used / 1e6, "lattice spectra:", 2 * ng * ng * (ng + 2) * 4 / 1e6, flush=True)
    assert used <= 2 * ng * ng * (ng + 2) * 4 + 8e6
