"""The work that programs have this library do, for timing and comparing builds.

Kinds of case, each through the public entry points:

  segment   a box is loaded from a checkpoint held in host memory, advanced by
            `steps` steps of the main loop (time step, drift, PP, PM, with the
            neutrino fluid where the box has one) and read back: what a host
            program does between two outputs.
  halofind  the halo catalogue of a resident box.
  power     the matter power spectrum of a resident box.
  ic        seeded initial conditions generated in device memory, read back.
  ensemble  a few boxes submitted to the serving engine and run to their end.

The inputs come from the seed alone, by torch on the GPU: a Gaussian field with
the library's linear spectrum, Zel'dovich displacements and velocities, and for
late times a share of the particles moved into NFW halos with virial velocity
dispersions.
"""
import ctypes
import math

import numpy as np
import torch

from cube_nufluid_amd import _lib, halo
from cube_nufluid_amd.checkpoint import BoxState
from cube_nufluid_amd.driver import Cube
from cube_nufluid_amd.ic import dgrow, ic_vsim2phys, linear_power, power_table, velocity_factor
from cube_nufluid_amd.params import NCELL, PI_F, BoxConfig
from cube_nufluid_amd.serving import run_ensemble

DEV = "cuda"
NSLAB = 1 << 24  # particles handled at a time by the host-side encoder


def listed():
    def seg(name, **kw):
        c = dict(name=name, kind="segment", nc=64, nnt=2, npd=128, izipx=2, izipv=2, pp=True, pp_range=1, z=3.0,
                 clump=0.0, nu=False, steps=8, mode=0, box=200.0)
        c.update(kw)
        return c
    return [
        # the smallest box of the serving mix, its steps replayed as graphs: launches and latency
        seg("serve 32^3 graph steps", nc=16, nnt=1, npd=32, box=50.0, z=2.0, steps=24, mode=2),
        # the plain PM test box of the reference's size, one call per phase, no pair force
        seg("box 64^3 pm only", nc=32, npd=64, box=100.0, pp=False, z=5.0, steps=16),
        # a serving box late in its run, one synchronisation per step
        seg("serve 128^3 late", nc=64, npd=128, z=0.6, clump=0.25, steps=8, mode=1),
        # 1-byte positions and velocities, particle lattice that no cell divides, narrow tiles, wider pair range
        seg("box 101^3 on 256^3 ragged", nc=64, nnt=8, npd=101, izipx=1, izipv=1, pp_range=2, z=1.0, clump=0.15, steps=8),
        # the middle configuration at an early time: nearly uniform cells, 1-byte positions
        seg("box 256^3 early", nc=128, nnt=4, npd=256, izipx=1, box=400.0, z=9.0, steps=8),
        # the same size at a late time: crowded cells, dense pair blocks
        seg("box 256^3 late", nc=128, nnt=4, npd=256, box=400.0, z=0.5, clump=0.3, steps=6),
        # CDM with the neutrino fluid, the fluids at 256^3, 128^3 and 64^3 cells
        seg("box 256^3 with neutrinos", nc=128, nnt=4, npd=256, box=250.0, z=9.0, nu=True, steps=4),
        # a production box at the time most of its steps are taken
        seg("box 512^3 clustered", nc=256, nnt=4, npd=512, box=500.0, z=1.1, clump=0.12, steps=8),
        # the catalogue at an output redshift
        dict(name="halos of 256^3", kind="halofind", nc=128, nnt=4, npd=256, izipx=2, izipv=2, z=0.0, clump=0.15, box=400.0),
        # the spectrum of the same kind of box on its 512^3 mesh
        dict(name="power of 256^3", kind="power", nc=128, nnt=4, npd=256, izipx=2, izipv=2, z=1.0, clump=0.2, box=400.0),
        # a start state for a run
        dict(name="start state 256^3", kind="ic", nc=128, nnt=4, npd=256, izipx=1, izipv=2, z=49.0, box=400.0),
        # small boxes served together from their start states
        dict(name="ensemble of small boxes", kind="ensemble", count=6, small=32, large=64, z=49.0, z_end=9.0, mode=2),
    ]


def draw(rng):
    kind = rng.choice(["segment"] * 7 + ["halofind", "power", "ic"])
    nc = rng.choice([16, 32, 64, 128])
    nnt = rng.choice([n for n in (1, 2, 4, 8) if nc // n >= 8])
    npd = int(round(math.exp(rng.uniform(math.log(1.2 * nc), math.log(2.2 * nc)))))
    z = round(math.exp(rng.uniform(math.log(1.3), math.log(20.0))) - 1.0, 3)
    clump = 0.0 if z > 3 else round(rng.uniform(0.05, 0.4), 3)
    c = dict(kind=kind, nc=nc, nnt=nnt, npd=npd, izipx=rng.choice([1, 2]), izipv=rng.choice([1, 2, 2]), z=z, clump=clump,
             box=round(1.5625 * npd * rng.uniform(0.7, 1.4), 2))
    if kind == "segment":
        nu = nc >= 32 and rng.random() < 0.2
        c.update(pp=rng.random() < 0.85, pp_range=rng.choice([1, 1, 1, 2, 3]), nu=nu, steps=rng.randint(3, 8),
                 mode=0 if nu else rng.choice([0, 0, 1, 2]))
        if nu:
            c.update(z=round(rng.uniform(4.0, 9.0), 3), clump=0.0)
    elif kind == "halofind":
        c.update(izipx=2, clump=round(rng.uniform(0.05, 0.2), 3), z=round(rng.uniform(0.0, 1.0), 3), npd=min(2 * nc, 256))
    elif kind == "ic":
        c.update(npd=2 * nc, z=round(rng.uniform(9.0, 99.0), 2))
        c.pop("clump")
    return c


# ------------------------------------------------------------------- inputs
def config(c):
    return BoxConfig(nc=c["nc"], nnt=c["nnt"], ncb=min(6, c["nc"] // c["nnt"]), izipx=c["izipx"], izipv=c["izipv"],
                     np_nc=2, box=c["box"], pp_on=c.get("pp", False), pp_range=c.get("pp_range", 1), z_i=c["z"],
                     m_nu_ev=0.1 / 3 if c.get("nu") else 0.0, z_i_nu=10.0)


def generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def wavenumbers(m):
    k = torch.fft.fftfreq(m, d=1.0 / m, device=DEV)
    kr = torch.fft.rfftfreq(m, d=1.0 / m, device=DEV)
    return k[:, None, None], k[None, :, None], kr[None, None, :]


def linear_field(cfg, m, a, seed):
    """The modes of the linear overdensity on an m^3 lattice."""
    kz, ky, kx = wavenumbers(m)
    kf = 2 * math.pi / cfg.box
    k2 = (kx * kx + ky * ky + kz * kz) * (kf * kf)
    k2[0, 0, 0] = 1.0
    lnk = np.linspace(math.log(1e-3), math.log(1e2), 4096)
    lnp = np.log(linear_power(cfg)(np.exp(lnk)) * dgrow(a, cfg.omega_m, cfg.omega_l) ** 2)
    tab = torch.tensor(lnp, dtype=torch.float32, device=DEV)
    t = (0.5 * torch.log(k2) - lnk[0]) / (lnk[1] - lnk[0])
    i = t.floor().clamp(0, 4094).long()
    t = t - i
    p = torch.exp(tab[i] * (1 - t) + tab[i + 1] * t)
    del i, t
    w = torch.fft.rfftn(torch.randn((m, m, m), generator=generator(seed, 1), device=DEV))
    w *= torch.sqrt(p * (m ** 3 / cfg.box ** 3))
    w[0, 0, 0] = 0
    return w, k2, kf


def displacement(cfg, w, k2, kf, m, e):
    """Component e (x, y, z) of the Zel'dovich displacement, in fine cells."""
    k = wavenumbers(m)[2 - e]
    fac = k * kf / k2
    fac = torch.where(k.abs() * 2 == m, torch.zeros((), device=DEV), fac)
    return torch.fft.irfftn(1j * fac * w, s=(m, m, m)) * (cfg.nf / cfg.box)


def nfw_radius(u, conc=6.0):
    """Radius over the virial radius at mass fraction u."""
    x = torch.linspace(0, conc, 4097, device=DEV, dtype=torch.float64)
    mu = torch.log1p(x) - x / (1 + x)
    mu = mu / mu[-1]
    i = torch.searchsorted(mu, u.double().contiguous()).clamp(1, 4096)
    f = (u - mu[i - 1]) / (mu[i] - mu[i - 1])
    return ((x[i - 1] + f * (x[i] - x[i - 1])) / conc).float()


def phase_space(cfg, c, seed):
    """Positions (fine cells) and velocities of npd^3 particles."""
    m, a = c["npd"], 1.0 / (1.0 + c["z"])
    n = m ** 3
    w, k2, kf = linear_field(cfg, m, a, seed)
    vfac = velocity_factor(cfg, a)
    pos = torch.empty((3, n), device=DEV)
    vel = torch.empty((3, n), device=DEV)
    for e in range(3):
        psi = displacement(cfg, w, k2, kf, m, e)
        # displacements of several cells only mix streams: late starts are cut to a few mean separations
        psi = psi * min(1.0, 2.0 * cfg.nf / m / max(1e-6, 3.0 * float(psi.std())))
        q = (torch.arange(m, device=DEV) + 0.5) * (cfg.nf / m)
        q = q.reshape([m if d == 2 - e else 1 for d in range(3)])
        pos[e] = (psi + q).reshape(-1)
        vel[e] = (psi * vfac).reshape(-1)
    del w, k2, psi
    share = c.get("clump", 0.0)
    if share > 0:
        g = generator(seed, 2)
        mmin, mmax = 20.0, min(3e3, 0.02 * n)  # a cluster of 10^15 solar masses at 1.5 Mpc/h a particle
        mean = mmin * math.log(mmax / mmin) / (1 - mmin / mmax)
        size = (mmin / (1 - torch.rand(max(1, int(share * n / mean)), generator=g, device=DEV) * (1 - mmin / mmax))).long()
        size = size[torch.cumsum(size, 0) <= int(0.9 * n)]
        total = int(size.sum())
        member = torch.randperm(n, generator=g, device=DEV)[:total]
        start = torch.cumsum(size, 0) - size
        owner = torch.repeat_interleave(torch.arange(len(size), device=DEV), size)
        mass = size.double() * (cfg.nf ** 3 / n)                          # in fine cells of mean density
        rvir = (3 * mass / (4 * math.pi * 200)) ** (1 / 3)
        sig = torch.sqrt(a * mass / (6 * math.pi * rvir) / 3).float()
        r = nfw_radius(torch.rand(total, generator=g, device=DEV)) * rvir.float()[owner]
        d = torch.randn((3, total), generator=g, device=DEV)
        d *= r / torch.sqrt((d * d).sum(0)).clamp(min=1e-6)
        first = member[start][owner]
        pos[:, member] = pos[:, first] + d
        vel[:, member] = vel[:, first] + sig[owner] * torch.randn((3, total), generator=g, device=DEV)
        del member, owner, first, r, d
    return pos, vel


def pinned(shape, dtype):
    return torch.empty(shape, dtype=dtype, pin_memory=True)


def box_state(cfg, c, seed):
    """The box in CUBE's checkpoint form, in pinned host memory."""
    pos, vel = phase_space(cfg, c, seed)
    n, nc, nt, nnt = pos.shape[1], cfg.nc, cfg.nt, cfg.nnt
    a = np.float32(1.0 / (1.0 + c["z"]))
    bits = 8 * cfg.izipx
    rank, code = None, torch.empty((3, n), dtype=torch.int32, device=DEV)
    for e in range(3):
        # whole position units: cells and codes by shifts
        u = torch.remainder(torch.floor(pos[e].double() * (2 ** bits / NCELL)).long(), nc << bits)
        cell = u >> bits
        code[e] = (u & ((1 << bits) - 1)).int()
        term = (cell // nt) * nnt ** e * nt ** 3 + (cell % nt) * nt ** e
        rank = term if rank is None else rank + term
    del pos, u, cell, term
    rank, order = torch.sort(rank, stable=True)
    n3 = nc ** 3
    rhoc = torch.bincount(rank, minlength=n3)
    # cell means by whole-number sums: the same for every order of adding
    vfield = torch.empty((n3, 3), device=DEV)
    res = torch.empty((3, n), device=DEV)
    for e in range(3):
        v = vel[e][order]
        s = torch.zeros(n3, dtype=torch.int64, device=DEV)
        s.index_add_(0, rank, torch.round(v.double() * 2 ** 24).long())
        vfield[:, e] = (s.double() / 2 ** 24 / rhoc.clamp(min=1)).float()
        res[e] = v - vfield[:, e][rank]
    vz_max, vall = float(vel[2].abs().max()), float(vel.abs().max())
    sigma = np.float32(math.sqrt(float((res.double() ** 2).sum()) / n / 3.0))
    coef = math.sqrt(float(PI_F) / 2) / (float(sigma) * 2.5)
    nv1 = float(2 ** (8 * cfg.izipv) - 1)
    xdt, vdt = (torch.int8, torch.int16)[cfg.izipx - 1], (torch.int8, torch.int16)[cfg.izipv - 1]
    out = [pinned((n, 3), xdt), pinned((n, 3), vdt), pinned((n,), torch.int32), pinned((n3,), torch.int32),
           pinned((n3, 3), torch.float32)]
    for i in range(0, n, NSLAB):
        j = min(n, i + NSLAB)
        x = code[:, order[i:j]]
        x = torch.where(x >= 1 << (bits - 1), x - (1 << bits), x).T
        out[0][i:j].copy_(x.contiguous().to(xdt))
        v = torch.round(nv1 / float(PI_F) * torch.atan(coef * res[:, i:j].double())).T
        out[1][i:j].copy_(v.contiguous().to(vdt))
        out[2][i:j].copy_((order[i:j] + 1).int())
    out[3].copy_(rhoc.int())
    out[4].copy_(vfield)
    sim = _lib.SimHeader()
    sim.nplocal = sim.npglobal = n
    sim.izipx, sim.izipv, sim.izipx_nu, sim.izipv_nu, sim.image = cfg.izipx, cfg.izipv, 2, 2, 1
    sim.nn, sim.nnt, sim.nt, sim.ncell, sim.ncb = 1, nnt, nt, NCELL, cfg.ncb
    sim.a = a
    sim.dt_pp = sim.dt_coarse = sim.dt_vmax_nu = 1000.0
    sim.dt_fine = 0.02
    sim.dt_vmax = 18.0 / vall
    sim.mass_p_cdm = cfg.mass_p(n)
    sim.box, sim.h0, sim.omega_m, sim.omega_l, sim.s8 = cfg.box, cfg.h0, cfg.omega_m, cfg.omega_l, cfg.sigma8
    sim.vsim2phys = ic_vsim2phys(cfg, a)
    sim.sigma_vi, sim.z_i, sim.z_i_nu, sim.vz_max = sigma, c["z"], cfg.z_i_nu, vz_max
    return BoxState(sim, *[t.numpy() for t in out])


def fluid_fields(cfg, c, cube, seed):
    """The three fluids from a smoothed linear field: density, momentum, energy."""
    a = 1.0 / (1.0 + c["z"])
    got = []
    for i in range(3):
        info = cube.nu_info(i)
        m = info["nc"]
        w, k2, kf = linear_field(cfg, m, a, seed + 17)
        l = torch.sqrt(k2) / (0.15 * (i + 1))
        w /= 1 + l + l * l
        f = torch.empty((5, m, m, m), device=DEV)
        f[0] = (1 + torch.fft.irfftn(w, s=(m, m, m))).clamp(min=0.3)
        f[0] /= f[0].mean()
        for e in range(3):
            f[1 + e] = f[0] * displacement(cfg, w, k2, kf, m, e) * velocity_factor(cfg, a)
        f[4] = f[0] * info["cs2"] / (5.0 / 3.0 - 1) + (f[1:4] ** 2).sum(0) / (2 * f[0])
        host = pinned((5, m, m, m), torch.float32)
        host.copy_(f)
        got.append(host.numpy())
        del w, k2, l, f
    return got


def buffers_like(st):
    return [pinned(x.shape, torch.from_numpy(x).dtype).numpy() for x in (st.xp, st.vp, st.pid, st.rhoc, st.vfield)]


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "ensemble":
        sizes = [c["small"] if i % 2 else c["large"] for i in range(c["count"])]
        return dict(case=c, requests=[dict(t=0.0, npd=s, seed=int(seed) * 100 + i, z_i=c["z"], z_f=c["z_end"])
                                      for i, s in enumerate(sizes)])
    cfg = config(c)
    s = dict(case=c, cfg=cfg)
    if c["kind"] == "ic":
        a = 1.0 / (1.0 + c["z"])
        s["cube"] = Cube.from_ic(cfg, int(seed), c["z"])
        lnk, lnp = power_table(cfg, a)
        ip = _lib.ICParams()
        ip.seed, ip.np_nc, ip.nk, ip.a, ip.box = int(seed), cfg.np_nc, len(lnk), a, cfg.box
        ip.vfac, ip.lnk, ip.lnp, ip.f_cdm = velocity_factor(cfg, a), _lib.ptr(lnk), _lib.ptr(lnp), cfg.f_cdm
        n, n3 = cfg.npart, cfg.nc ** 3
        dts = (torch.int8, torch.int16)
        s.update(ip=ip, table=(lnk, lnp),
                 out=[pinned((n, 3), dts[c["izipx"] - 1]).numpy(), pinned((n, 3), dts[c["izipv"] - 1]).numpy(),
                      pinned((n,), torch.int32).numpy(), pinned((n3,), torch.int32).numpy(),
                      pinned((n3, 3), torch.float32).numpy()])
        return s
    st = box_state(cfg, c, seed)
    if c["kind"] == "halofind":
        cat = halo.cube_halo_catalog()
        cat.max_halos, cat.max_pid_words = st.sim.nplocal // 100, st.sim.nplocal // 2
        s["halos"] = np.zeros((cat.max_halos, halo.HALO_RECORD_FLOATS), dtype=np.float32)
        s["words"] = np.zeros(cat.max_pid_words, dtype=np.int32)
        cat.halos, cat.pid_words = s["halos"].ctypes.data, s["words"].ctypes.data
        s["cat"], s["hp"] = cat, halo.params_struct(halo.HaloParams().for_box(cfg, None, st.sim))
    torch.cuda.empty_cache()  # the library allocates beside torch
    s["cube"] = cube = Cube(cfg, st, np_max=st.sim.nplocal, z_checkpoints=[c["z"], -0.5])
    s["state"] = st
    if c["kind"] == "segment":
        s["out"] = buffers_like(st)
        _lib.check(cube.lib, cube.h, cube.lib.cube_set_step_mode(cube.h, c["mode"]))
        s["z"] = np.array([c["z"], -0.5], dtype=np.float32)
        if c["nu"]:
            cube.nu_init(m_ev=cfg.m_nu_ev, f_neu=cfg.f_neu, z_i_nu=cfg.z_i_nu)
            s["fluids"] = fluid_fields(cfg, c, cube, seed)
            s["fluids_out"] = [pinned(f.shape, torch.float32).numpy() for f in s["fluids"]]
            torch.cuda.empty_cache()
    return s


# --------------------------------------------------------------------- runs
def run_segment(s):
    cube, c = s["cube"], s["case"]
    lib, h = cube.lib, cube.h
    cube.upload(s["state"])
    clock = _lib.CubeClock()
    _lib.check(lib, h, lib.cube_clock_init(ctypes.byref(clock), _lib.ptr(s["z"]), len(s["z"])))
    if c["nu"]:
        for i, f in enumerate(s["fluids"]):
            cube.nu_set(i, f)
        cube.nu_seed_dt()
        clock.dt_neu = float(cube.dt_neu)
    for _ in range(c["steps"]):
        _lib.check(lib, h, lib.cube_step(h, ctypes.byref(clock)))
    sim, out = _lib.SimHeader(), s["out"]
    _lib.check(lib, h, lib.cube_download_state(h, ctypes.byref(sim), *[_lib.ptr(x) for x in out]))
    got = dict(zip(("xp", "vp", "pid", "rhoc", "vfield"), out))
    got.update(a=clock.a, t=clock.t, dt=clock.dt, istep=clock.istep, sigma_vi=sim.sigma_vi, vz_max=sim.vz_max)
    if c["nu"]:
        for i, f in enumerate(s["fluids_out"]):
            _lib.check(lib, h, lib.cube_nu_get_fluid(h, i, _lib.ptr(f)))
            got["fluid%d" % i] = f
        got["dt_neu"] = clock.dt_neu
    return got


def run(s):
    c = s["case"]
    if c["kind"] == "segment":
        return run_segment(s)
    if c["kind"] == "halofind":
        cube, cat = s["cube"], s["cat"]
        _lib.check(cube.lib, cube.h, cube.lib.cube_halofind(cube.h, ctypes.byref(s["hp"]), ctypes.byref(cat)))
        return dict(halos=s["halos"], pid_words=s["words"], nhalo=cat.nhalo, npid_words=cat.npid_words, npeaks=cat.npeaks,
                    nprocessed=cat.nprocessed)
    if c["kind"] == "power":
        k, d2, modes = s["cube"].power_spectrum()
        return dict(k=k, d2=d2, modes=modes)
    if c["kind"] == "ic":
        lib, h, sim = s["cube"].lib, s["cube"].h, _lib.SimHeader()
        _lib.check(lib, h, lib.cube_ic_zeldovich(h, ctypes.byref(s["ip"]), ctypes.byref(sim)))
        _lib.check(lib, h, lib.cube_download_state(h, None, *[_lib.ptr(x) for x in s["out"]]))
        got = dict(zip(("xp", "vp", "pid", "rhoc", "vfield"), s["out"]))
        got.update(sigma_vi=sim.sigma_vi, vz_max=sim.vz_max)
        return got
    res = run_ensemble(s["requests"], max_live=16, step_mode=c["mode"])["results"]
    res = sorted(res, key=lambda r: r["seed"])
    return dict(steps=np.array([r["steps"] for r in res]), a=np.array([r["a_final"] for r in res], dtype=np.float32),
                state=np.array([r["hash"] for r in res], dtype=np.uint64).view(np.int64))


# --------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass that no arrangement saves.  A step reads
    and writes the particles once; its fine mesh is transformed once forward and
    three times back, and a transform of a mesh beyond the on-chip memory reads
    and writes it twice (8 bytes a node each time); 2.5 N^3 log2(N^3) operations a
    transform and some 300 a particle.  A load and a read-back move the state."""
    c = dict(case)
    if c["kind"] == "ensemble":
        w = {"bytes": 0.0, "flops": 0.0}
        for i in range(c["count"]):
            m = c["small"] if i % 2 else c["large"]
            one = work(dict(kind="segment", nc=m // 2, npd=m, izipx=2, izipv=2, steps=24, nu=False))
            w = {k: w[k] + one[k] for k in w}
        return w
    n, nc = float(c["npd"]) ** 3, float(c["nc"])
    mf, part, cells = (4 * nc) ** 3, 3.0 * (c["izipx"] + c["izipv"]) + 4, 16 * nc ** 3
    fft = 2.5 * mf * math.log2(mf)
    state = part * n + cells
    if c["kind"] == "segment":
        step = 2 * state + 4 * 2 * 8 * mf
        flops = 4 * fft + 300 * n
        if c["nu"]:
            fluid = sum(20.0 * (4 * nc / d) ** 3 for d in (2, 4, 8))
            step, state = step + 4 * fluid, state + fluid
        return {"bytes": c["steps"] * step + 2 * state, "flops": c["steps"] * flops}
    if c["kind"] == "halofind":
        return {"bytes": 3 * c["izipx"] * n + 8 * mf, "flops": 50 * n + 30 * mf}
    if c["kind"] == "power":
        return {"bytes": 3 * c["izipx"] * n + 16 * mf, "flops": 50 * n + fft + 20 * mf}
    return {"bytes": state + 4 * 2 * 8 * n, "flops": 4 * 2.5 * n * math.log2(n) + 100 * n}


# -------------------------------------------------------------------- exact
def exact(case, seed):
    """The power spectrum in 64 bits: CIC density, transform, window, bins.

    A segment's state is whole codes whose every step rounds them, and a
    catalogue's members are whole numbers: those have no 64-bit value.  Nor has
    the vfield of start states, means of velocities rounded to codes."""
    c = dict(case)
    if c["kind"] != "power":
        return None
    cfg = config(c)
    st = box_state(cfg, c, seed)
    ng, nc, nt, nnt = cfg.nf, cfg.nc, cfg.nt, cfg.nnt
    r = torch.repeat_interleave(torch.arange(nc ** 3, device=DEV), torch.from_numpy(st.rhoc).to(DEV).long())
    t, l = r // nt ** 3, r % nt ** 3
    bits = 8 * cfg.izipx
    i0, w1 = [], []
    for e in range(3):
        cell = (t // nnt ** e % nnt) * nt + l // nt ** e % nt
        u = torch.from_numpy(np.ascontiguousarray(st.xp[:, e])).to(DEV).long() & ((1 << bits) - 1)
        x = NCELL * (cell + (u.double() + 0.5) / 2.0 ** bits)
        i0.append(torch.floor(x).long())
        w1.append(1.0 - (x - torch.floor(x)))
    rho = torch.zeros(ng ** 3, dtype=torch.float64, device=DEV)
    for corner in range(8):
        o = [corner & 1, corner >> 1 & 1, corner >> 2]
        w, at = 1.0, 0
        for e in range(3):
            w = w * (1.0 - w1[e] if o[e] else w1[e])
            at = at + (i0[e] + o[e]) % ng * ng ** e
        rho.index_add_(0, at, w)
    del r, t, l, i0, w1, w, at
    rho = rho.reshape(ng, ng, ng)
    modes = torch.fft.rfftn(rho / rho.mean() - 1.0) / ng ** 3
    nyq = ng // 2
    q = torch.fft.fftfreq(ng, d=1.0 / ng, device=DEV, dtype=torch.float64)
    i = torch.arange(ng, device=DEV)
    kz, ky, kx = i[:, None, None], i[None, :, None], i[None, None, :nyq + 1]
    edge = (kx == 0) | (kx == nyq)
    keep = ~((kx == 0) & (ky == 0) & (kz == 0)) & ~(edge & (ky > nyq)) & ~(edge & ((ky == 0) | (ky == nyq)) & (kz > nyq))
    sinc = torch.where(q == 0, 1.0, torch.sin(math.pi * q / ng) / torch.where(q == 0, 1.0, math.pi * q / ng))
    k2 = q[:, None, None] ** 2 + q[None, :, None] ** 2 + q[None, None, :nyq + 1] ** 2
    # the bin edges are the reference's, in 32 bits
    kr = torch.sqrt(k2.float())
    ib = torch.floor(kr + 0.5).long()
    win = sinc[:, None, None] * sinc[None, :, None] * sinc[None, None, :nyq + 1]
    amp = modes.abs() ** 2 / win ** 4 * 4 * math.pi * kr.double() ** 3
    nbin = int(np.rint(nyq * np.sqrt(3.0)))
    ib = torch.where(keep, ib, 0).reshape(-1)
    sums = [torch.zeros(nbin + 2, dtype=torch.float64, device=DEV).index_add_(0, ib.clamp(max=nbin + 1), x.reshape(-1))
            for x in (torch.ones_like(amp), kr.double(), amp)]
    n, ks, d2 = [x[1:nbin + 1].cpu().numpy() for x in sums]
    n1 = np.maximum(n, 1)
    return dict(k=ks / n1 * 2 * np.pi / cfg.box, d2=d2 / n1, modes=n)
