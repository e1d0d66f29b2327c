"""Performance cases: the work a user of this package has one MI355X do.

A case is one pass through the public entry points (colore_amd.lib), from what
a program has in hand (a parsed parameter file with its tables, a context, its
host buffers) to the outputs on the host.  Grid sizes, cosmology, populations,
source planes and shells are those of colore_amd.inputs.CONFIGS and of the
tests, at sizes from 64^3 to 1024^3.

  kind        one pass
  chain       Gaussian fields, lognormal + shell norms, every population's
              sources, a convergence map, the catalogues on the host: one mock
  maps        Gaussian fields, density + shell norms, convergence and ISW
              maps and (optionally) a custom map: one lensing mock
  sources     the sources of a given density, catalogues on the host
  beams       the line-of-sight pass of a catalogue: RSD, shear, convergence,
              deflection per source
  skewers     density and velocity skewers of a (quasar) catalogue
  imap        21cm intensity maps of a given density
  lpt         Gaussian fields, 1LPT or 2LPT density, shell norms, custom map
"""
import functools
import math
import tempfile

import numpy as np
import torch

from colore_amd import inputs, lib

NSIDE_BASE = 2


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest whole mock: launches, synchronisations and small copies
        dict(name="chain_64", kind="chain", config="C2", n_grid=64, z_max=1.2, r_smooth=2.0, density=0.005,
             nside=32),
        # an odd (3 2^n) grid with three populations, one of each bias model
        dict(name="chain_192", kind="chain", config="C3", n_grid=192, z_max=1.6, r_smooth=2.0, density=0.02,
             nside=64),
        # the two-population configuration as it stands: 1.3e7 sources
        dict(name="chain_512", kind="chain", config="C2", n_grid=512, z_max=1.2, r_smooth=2.0, density=1.0,
             nside=256),
        # a mid-size lensing mock, only the density smoothed, with a custom map
        dict(name="maps_256", kind="maps", config="C2", n_grid=256, z_max=1.2, r_smooth=2.0, smooth_potential=False,
             density_type="lognormal", nside=256, custom=True),
        # the flagship grid with its three source planes: convergence and ISW
        dict(name="maps_1024", kind="maps", config="C3", n_grid=1024, z_max=1.6, r_smooth=1.0, smooth_potential=True,
             density_type="lognormal", nside=512, custom=False),
        # the flagship grid's three populations at a tenth of their densities
        # (1e-5 .. 1e-4 per (Mpc/h)^3, spectroscopic samples): 2.7e6 sources
        dict(name="sources_1024", kind="sources", config="C3", n_grid=1024, z_max=1.6, density=0.1),
        # a denser sampling on a small grid: several sources in many cells
        dict(name="sources_128", kind="sources", config="C1", n_grid=128, z_max=0.5, density=0.3),
        # shear, convergence and deflection of 1e6 lensed sources
        dict(name="beams_512", kind="beams", config="C2", n_grid=512, z_max=1.2, density=0.1),
        # Lyman-alpha skewers of 3e4 quasars
        dict(name="skewers_384", kind="skewers", config="C2", n_grid=384, z_max=1.2, density=0.003,
             gaussian=False),
        # 21cm shells, a third of the flagship's bands
        dict(name="imap_256", kind="imap", config="C3", n_grid=256, z_max=1.6, nside=128, bands=24),
        # Lagrangian densities: first order on a mid-size grid ...
        dict(name="lpt1_512", kind="lpt", config="C2", n_grid=512, z_max=1.2, r_smooth=2.0, order=1, interp=1,
             nside=128),
        # ... and second order with the wider kernel on a small one
        dict(name="lpt2_128", kind="lpt", config="C2", n_grid=128, z_max=1.2, r_smooth=2.0, order=2, interp=2,
             nside=64),
    ]


def _logu(rng, lo, hi):
    return float("%.4g" % math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["chain", "chain", "maps", "maps", "sources", "beams", "skewers", "imap", "lpt"])
    config = rng.choice(["C2", "C3"])
    c = dict(kind=kind, config=config, z_max=round(rng.uniform(0.9, 1.2) if config == "C2" else rng.uniform(1.0, 1.6), 3))
    if kind == "chain":
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384, 512])
        c.update(r_smooth=round(rng.uniform(0.5, 4.0), 2), density=_logu(rng, 0.002, 0.5), nside=rng.choice([32, 64, 128, 256]))
    elif kind == "maps":
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384, 512, 1024])
        c.update(r_smooth=round(rng.uniform(1.0, 4.0), 2), smooth_potential=rng.random() < 0.7,
                 density_type=rng.choice(["lognormal", "lognormal", "clip"]), nside=rng.choice([32, 64, 128, 256, 512]),
                 custom=rng.random() < 0.5 and c["n_grid"] < 1024)
    elif kind == "sources":
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384, 512])
        c["density"] = _logu(rng, 0.002, 0.5)
    elif kind == "beams":
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384, 512])
        c["density"] = _logu(rng, 0.002, 0.1)
    elif kind == "skewers":
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384])
        c["density"] = _logu(rng, 0.0003, 0.003)
        c["gaussian"] = rng.random() < 0.4
    elif kind == "imap":
        c["config"], c["z_max"] = "C3", round(rng.uniform(1.0, 1.6), 3)
        c["n_grid"] = rng.choice([64, 128, 192, 256])
        c.update(nside=rng.choice([16, 32, 64, 128]), bands=rng.randint(5, 24))
    else:
        order = rng.choice([1, 2])
        c["n_grid"] = rng.choice([64, 128, 192, 256, 384] if order == 1 else [64, 128, 192])
        c.update(r_smooth=round(rng.uniform(2.0, 4.0), 2), order=order, interp=rng.choice([1, 2]),
                 nside=rng.choice([32, 64, 128]))
    return c


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _parsed(config, n_grid, z_max, r_smooth, density, bands, nside_imap):
    """The parsed parameter file of a configuration, its populations' number
    densities scaled by `density`."""
    pops = []
    for nz, bz, model in inputs.CONFIGS[config]["srcs"]:
        nz = list(nz)
        nz[3] = nz[3] * density
        pops.append((tuple(nz), bz, model))
    with tempfile.TemporaryDirectory() as d:
        return lib.Run(inputs.write_config(config, d, n_grid=n_grid, z_max=z_max, r_smooth=r_smooth, populations=pops,
                                           with_maps=bool(bands), imap_bands=bands or None,
                                           imap_nside=nside_imap or None))


def _run_of(case):
    return _parsed(case["config"], case["n_grid"], case["z_max"], case.get("r_smooth", 2.0), case.get("density", 0.1),
                   case.get("bands", 0), case["nside"] if case["kind"] == "imap" else 0)


def _seed32(seed):
    return (seed * 2654435761 + 12345) % (1 << 32)


def _planes(run, z_max):
    """Source planes at the configurations' z = 0.5, 1.0, 1.5 inside the box."""
    host = lib.load_host()
    return np.array([host.clr_run_r_of_z(run.h, z) for z in (0.5, 1.0, 1.5) if z <= z_max])


def _tracers(case, run):
    """(kind, index, model, amplitude table, bias table) in the call order."""
    out = []
    if case["kind"] == "imap":
        amp, bz, model = run.tracer(lib.CLR_TRACER_IMAP, 0)
        return [(lib.CLR_TRACER_IMAP, 0, model, amp, bz)]
    npop = int(run.scalar("n_srcs"))
    if case["kind"] in ("beams", "skewers", "lpt"):
        npop = 1
    for i in range(npop):
        amp, bz, model = run.tracer(lib.CLR_TRACER_SRCS, i)
        out.append((lib.CLR_TRACER_SRCS, i, model, amp, bz))
    if case.get("custom") or case["kind"] == "lpt":
        # a projected map with the first population's n(r) and b(r) as kernel and bias
        out.append((lib.CLR_TRACER_CSTM, 0, 0, out[0][3], out[0][4]))
    return out


def _expected(run, amp):
    """Expected number of sources of a population with n(r) = amp (per (Mpc/h)^3)."""
    r = run.table_arrays()["r"]
    half = 0.5 * run.scalar("l_box") + 20
    w = np.where(r < half, amp * 4 * math.pi * r ** 2, 0.0)
    return float(np.trapezoid(w, r))


def _capacity(run, amp):
    """Rows of a catalogue buffer of that population."""
    return int(1.2 * _expected(run, amp)) + 4096


def _zeroed(shape, dtype=np.float32):
    """A page-locked host buffer; rows past a catalogue's end stay zero."""
    a = lib.pinned_empty(shape, dtype)
    a.fill(0)
    return a


def _gaussian_grid(case, run, seed):
    """Random density (lognormal on the lightcone) and potential grids of the
    configuration's power spectrum, float32[N][N][N+2] on the GPU."""
    ta = run.table_arrays()
    N, L = case["n_grid"], run.scalar("l_box")
    dev = torch.device("cuda", 0)
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed + 977)
    f = torch.fft.rfftn(torch.randn((N, N, N), generator=gen, device=dev))
    k1 = torch.fft.fftfreq(N, 1.0 / N, device=dev) * (2 * math.pi / L)
    kx = torch.arange(N // 2 + 1, device=dev) * (2 * math.pi / L)
    k2 = k1[:, None, None] ** 2 + k1[None, :, None] ** 2 + kx[None, None, :] ** 2
    k2[0, 0, 0] = 1.0
    lk = (0.5 * torch.log10(k2) - ta["logkmin"]) * ta["idlogk"]
    pk = torch.tensor(ta["pk"], dtype=torch.float32, device=dev)
    i = lk.long().clamp_(0, ta["numk"] - 2)
    p = pk[i] + (lk - i) * (pk[i + 1] - pk[i])
    rs = run.scalar("r_smooth")
    del i, lk
    f *= torch.sqrt(p * (N / L) ** 3) * torch.exp(-0.5 * rs * rs * k2)
    f[0, 0, 0] = 0
    del p
    g = torch.fft.irfftn(f, s=(N, N, N))
    sigma2 = float(g.double().var(correction=0))
    f *= -ta["prefac_lensing"] / k2
    phi = torch.fft.irfftn(f, s=(N, N, N))
    del f, k2
    x = torch.arange(N, device=dev) * (L / N) - 0.5 * L
    r = torch.sqrt(x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2)
    D = torch.tensor(ta["d1"], dtype=torch.float32, device=dev)
    i = (r * ta["glob_idr"]).long().clamp_(0, len(D) - 1)
    d = D[i]
    del r, i
    g = torch.expm1(d * (g - 0.5 * d * sigma2))
    return g, phi, sigma2


def _upload(ctx, which, g):
    """A grid of the GPU through page-locked host memory (clr_upload_grid takes host memory)."""
    host = torch.empty(ctx.padded_shape, pin_memory=True)
    host.copy_(torch.nn.functional.pad(g, (0, 2)))
    ctx.upload_grid(which, host.numpy())


def prepare(case, seed):
    run = _run_of(case)
    N = case["n_grid"]
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    tracers = _tracers(case, run)
    for kind, i, model, amp, bz in tracers:
        ctx.set_tracer(kind, i, model, amp, bz)
    kind = case["kind"]
    s = dict(case=case, run=run, ctx=ctx, seed=_seed32(seed), ntr=len(tracers), rs=run.scalar("r_smooth"),
             npop=sum(t[0] == lib.CLR_TRACER_SRCS for t in tracers))
    if kind in ("sources", "beams", "skewers", "imap"):
        dens, phi, s["sigma2"] = _gaussian_grid(case, run, seed)
        _upload(ctx, lib.CLR_GRID_DENS, dens)
        _upload(ctx, lib.CLR_GRID_NPOT, phi)
        del dens, phi
        torch.cuda.empty_cache()
        ctx.declare_grids(s["sigma2"], True)
        ctx.shell_norms(lognormal_fused=False, sigma2=s["sigma2"], ntracers=len(tracers))
    if kind in ("chain", "sources"):
        # host buffers of the catalogues, filled again by every realisation
        caps = [_capacity(run, t[3]) for t in tracers]
        s["cat"] = [(_zeroed((cap, 4)), _zeroed((cap,), np.int32)) for cap in caps]
    if kind in ("chain", "maps"):
        s["r_src"] = _planes(run, case["z_max"])
        if kind == "chain":
            s["r_src"] = s["r_src"][-1:]
        shape = (len(s["r_src"]), 12 * case["nside"] ** 2)
        s["kappa"] = lib.pinned_empty(shape)
        if kind == "maps":
            s["isw"] = lib.pinned_empty(shape)
    if kind in ("beams", "skewers"):
        n = s["n"] = ctx.sample_sources(0, s["seed"], NSIDE_BASE)
        cap = max(n, _capacity(run, tracers[0][3]))
        if kind == "beams":
            s["a2r"] = np.ascontiguousarray(run.r_a2r())
            s["dz"], s["lens"] = _zeroed((cap,)), _zeroed((cap, 5))
        else:
            s["dg"], s["v"] = _zeroed((cap, N // 2)), _zeroed((cap, N // 2))
    if kind == "imap":
        s["nside"], s["r0"], s["rf"] = run.imap_shells(0)
        shape = (len(s["r0"]), 12 * s["nside"] ** 2)
        s["data"], s["nadd"] = lib.pinned_empty(shape), lib.pinned_empty(shape, np.int32)
    return s


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------
def _chk(ctx, rc):
    if rc:
        raise RuntimeError(ctx.lib.clr_last_error(ctx.h).decode())


def _f(a):
    return lib.ptr(a, lib.ctypes.c_float)


def _i(a):
    return lib.ptr(a, lib.ctypes.c_int32)


def _catalogues(s):
    """Every population's catalogue, copied into the program's host buffers."""
    ctx, out = s["ctx"], []
    for i in range(s["npop"]):
        pos, ipix = s["cat"][i]
        n = ctx.catalogue_size(i)
        if n > len(pos):
            pos, ipix = s["cat"][i] = _zeroed((n, 4)), _zeroed((n,), np.int32)
        _chk(ctx, ctx.lib.clr_fetch_sources(ctx.h, i, _f(pos), _i(ipix), n))
        out.append((n, pos, ipix))
    return out


def _norms(s, fused, sigma2):
    """The shell sums and every tracer's normalisation table."""
    ctx = s["ctx"]
    _, cnt, zs, sums = ctx.shell_norms(lognormal_fused=fused, sigma2=sigma2, ntracers=s["ntr"])
    tabs = [ctx.norm_table(lib.CLR_TRACER_SRCS, i)[0] for i in range(s["npop"])]
    if s["ntr"] > s["npop"]:
        tabs.append(ctx.norm_table(lib.CLR_TRACER_CSTM, 0)[0])
    return [cnt, zs, sums, np.stack(tabs)]


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "chain":
        s2 = ctx.gaussian_fields(s["seed"], s["rs"], True)
        norms = _norms(s, True, s2)
        ctx.sample_sources(-1, s["seed"], NSIDE_BASE)
        return dict(sigma2=s2, norms=norms, kappa=ctx.kappa(case["nside"], s["r_src"], out=s["kappa"]),
                    catalogues=_catalogues(s))
    if kind == "maps":
        s2 = ctx.gaussian_fields(s["seed"], s["rs"], case["smooth_potential"])
        fused = case["density_type"] == "lognormal"
        if not fused:
            ctx.density(lib.CLR_DENS_CLIP, s2)
        out = dict(sigma2=s2, norms=_norms(s, fused, s2), kappa=ctx.kappa(case["nside"], s["r_src"], out=s["kappa"]),
                   isw=ctx.isw(case["nside"], s["r_src"], out=s["isw"]))
        if case["custom"]:
            out["custom"] = ctx.custom_map(0, case["nside"])
        return out
    if kind == "sources":
        ctx.sample_sources(-1, s["seed"], NSIDE_BASE)
        return _catalogues(s)
    if kind == "beams":
        _chk(ctx, ctx.lib.clr_source_beams(ctx.h, 0, lib.ptr(s["a2r"]), _f(s["dz"]), _f(s["lens"]), s["n"]))
        return [s["dz"], s["lens"]]
    if kind == "skewers":
        _chk(ctx, ctx.lib.clr_source_skewers(ctx.h, 0, int(case["gaussian"]), s["sigma2"], _f(s["dg"]), _f(s["v"]),
                                             s["n"]))
        return [s["dg"], s["v"]]
    if kind == "imap":
        _chk(ctx, ctx.lib.clr_imap(ctx.h, 0, s["nside"], len(s["r0"]), lib.ptr(s["r0"]), lib.ptr(s["rf"]),
                                   _f(s["data"]), _i(s["nadd"])))
        return [s["data"], s["nadd"]]
    s2 = ctx.gaussian_fields(s["seed"], s["rs"], True)
    ctx.lpt_density(case["interp"], case["order"])
    norms = _norms(s, False, s2)
    return dict(sigma2=s2, norms=norms, custom=ctx.custom_map(0, case["nside"]))


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the final grids written or the given grids read once, and the
    outputs written once.  Operations: 2.5 n log2 n per real transform, a few
    tens per cell, source, map step or sub-point for the rest."""
    kind, N = case["kind"], case["n_grid"]
    cells = float(N) ** 3
    fft = 2.5 * cells * 3 * math.log2(N)
    npix = 12.0 * case.get("nside", 0) ** 2
    run = _run_of(case)
    nsrc = [_expected(run, t[3]) for t in _tracers(case, run) if t[0] == lib.CLR_TRACER_SRCS]
    if kind == "chain":
        return dict(bytes=8 * cells + 20 * sum(nsrc) + 4 * npix,
                    flops=2 * fft + 150 * cells + 100 * sum(nsrc) + 40 * npix * N / 2)
    if kind == "maps":
        npl = len(_planes(run, case["z_max"]))
        return dict(bytes=8 * cells + (8 * npl + 4 * case["custom"]) * npix,
                    flops=2 * fft + 150 * cells + (50 + 40 * case["custom"]) * npix * N / 2)
    if kind == "sources":
        return dict(bytes=4 * cells + 44 * sum(nsrc), flops=30 * cells * len(nsrc) + 100 * sum(nsrc))
    if kind == "beams":
        return dict(bytes=4 * cells + 40 * nsrc[0], flops=60 * nsrc[0] * N / 3)
    if kind == "skewers":
        return dict(bytes=8 * cells + 16 * nsrc[0] + 8 * nsrc[0] * N / 2, flops=80 * nsrc[0] * N / 3)
    if kind == "imap":
        return dict(bytes=8 * cells + 8 * case["bands"] * npix, flops=60 * cells)
    nfft = 1 + 1 + 3 + (10 if case["order"] == 2 else 0)
    return dict(bytes=4 * cells + 4 * npix, flops=nfft * fft + 100 * cells + 40 * npix * N / 2)


# ---------------------------------------------------------------------------
# exact: the same results in 64 bits with torch
# ---------------------------------------------------------------------------
_M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, k0, k1=0x436F4C52):
    """Philox4x32-10 (Salmon et al. 2011) on int64 tensors or ints holding 32-bit words."""
    def mul(m, x):
        # 32 x 32 -> (high, low) words, through 16-bit halves of x: int64 has no room for the whole product
        a, b = m * (x >> 16), m * (x & 0xFFFF)
        t = a + (b >> 16)
        return (t >> 16) & _M32, ((t & 0xFFFF) << 16) | (b & 0xFFFF)
    for i in range(10):
        if i:
            k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
    return c0, c1, c2, c3


class _Exact:
    def __init__(self, case):
        self.case, self.run = case, _run_of(case)
        self.dev = torch.device("cuda", 0)
        ta = self.ta = self.run.table_arrays()
        self.N, self.L = case["n_grid"], self.run.scalar("l_box")
        self.dx = self.L / self.N
        self.r_arr = self.t(ta["r"])
        self.nr = self.N // 2
        self.dr = ta["r_max"] / self.nr

    def t(self, a):
        return torch.as_tensor(np.asarray(a), dtype=torch.float64, device=self.dev)

    def tab(self, name, r, f0, ff=None):
        """Linear interpolation of an r-table with its edge values."""
        f = self.t(self.ta[name]) if isinstance(name, str) else self.t(name)
        i = (r * self.ta["glob_idr"]).long().clamp_(0, len(f) - 2)
        v = f[i] + (f[i + 1] - f[i]) * (r - self.r_arr[i]) * self.ta["glob_idr"]
        v = torch.where(r <= 0, torch.full_like(v, float(f[0]) if f0 is None else f0), v)
        return torch.where(r >= self.r_arr[-1], torch.full_like(v, float(f[-1]) if ff is None else ff), v)

    def D(self, r):
        return self.tab("d1", r, 1.0)

    def z(self, r):
        return self.tab("z", r, 0.0)

    def axis(self):
        return torch.arange(self.N, device=self.dev, dtype=torch.float64) * self.dx - 0.5 * self.L

    def radius(self, iz):
        """Radii of the plane(s) iz (slice), [nz][N][N]."""
        x = self.axis()
        return torch.sqrt(x[None, None, :] ** 2 + x[None, :, None] ** 2 + x[iz][:, None, None] ** 2)

    def chunks(self):
        n = max(1, min(self.N, (1 << 25) // (self.N * self.N)))
        return [slice(a, min(self.N, a + n)) for a in range(0, self.N, n)]

    # -- fields ------------------------------------------------------------
    def fields(self, seed, rs, smooth_potential):
        N, L, ta = self.N, self.L, self.ta
        NH, dk = N // 2 + 1, 2 * math.pi / L
        spec = torch.empty((N, N, NH), dtype=torch.complex128, device=self.dev)
        kx = torch.arange(NH, device=self.dev)
        fy = torch.fft.fftfreq(N, 1.0 / N, device=self.dev).abs().long()
        pk = self.t(ta["pk"])
        logk = self.t(ta["logk"])
        ky = torch.arange(N, device=self.dev)
        step = max(1, (1 << 24) // (N * NH))
        for a in range(0, N // 2, step):
            kz = torch.arange(a, min(N // 2, a + step), device=self.dev)
            site = kx[None, None, :] + NH * (ky[None, :, None] + N * kz[:, None, None])
            w = _philox(site & _M32, site >> 32, 0, 0, seed)
            for h in (0, 1):
                fz = fy[kz + h * (N // 2)]
                k2 = dk * dk * (kx[None, None, :] ** 2 + fy[None, :, None] ** 2 + fz[:, None, None] ** 2).double()
                k2 = torch.where(k2 == 0, torch.ones_like(k2), k2)
                lk = 0.5 * torch.log10(k2)
                ik = ((lk - ta["logkmin"]) * ta["idlogk"]).long()
                j = ik.clamp(0, ta["numk"] - 2)
                p = pk[j] + (lk - logk[j]) * (pk[j + 1] - pk[j]) * ta["idlogk"]
                p = torch.where(lk < ta["logkmin"], pk[0] * 10 ** (ta["ns"] * (lk - ta["logkmin"])), p)
                p = torch.where(ik >= ta["numk"] - 1, pk[-1] * 10 ** (-3 * (lk - ta["logkmax"])), p)
                m = torch.sqrt(-p / dk ** 3 * torch.log1p(-w[2 * h + 1].double() / 2.0 ** 32))
                spec[kz + h * (N // 2)] = torch.polar(m, 2 * math.pi * w[2 * h].double() / 2.0 ** 32)
        spec[0, 0, 0] = 0

        def filtered(smooth, phi):
            out = spec.clone()
            for sl in self.chunks():
                k2 = dk * dk * (kx[None, None, :] ** 2 + fy[None, :, None] ** 2 + fy[sl][:, None, None] ** 2).double()
                f = torch.exp(-0.5 * rs * rs * k2) if smooth else torch.ones_like(k2)
                if phi:
                    f *= -ta["prefac_lensing"] / torch.where(k2 == 0, torch.ones_like(k2), k2)
                out[sl] *= f
            return self.c2r(out) * (math.sqrt(2 * math.pi) / L) ** 3

        dens = filtered(rs > 0, False)
        phi = filtered(rs > 0 and smooth_potential, True)
        return dens, phi

    def c2r(self, h):
        """Unnormalised complex-to-real transform: z and y, then x with the
        imaginary parts of the kx = 0 and N/2 planes dropped."""
        for ax in (0, 1):
            h = torch.fft.ifft(h, dim=ax, norm="forward")
        h[:, :, 0].imag.zero_()
        h[:, :, -1].imag.zero_()
        return torch.fft.irfft(h, n=self.N, dim=2, norm="forward")

    def density(self, g, sigma2, clip):
        for sl in self.chunks():
            D = self.D(self.radius(sl))
            g[sl] = torch.clamp(1 + D * g[sl], min=0) - 1 if clip else torch.expm1(D * (g[sl] - 0.5 * D * sigma2))
        return g

    def lpt(self, g, order, interp):
        N, dk = self.N, 2 * math.pi / self.L
        k1 = torch.fft.fftfreq(N, 1.0 / N, device=self.dev, dtype=torch.float64)
        k1[N // 2] = N // 2
        k1 = k1 * dk
        kx = torch.arange(N // 2 + 1, device=self.dev, dtype=torch.float64) * dk
        kv = [kx[None, None, :], k1[None, :, None], k1[:, None, None]]
        k2 = (kv[0] ** 2 + kv[1] ** 2 + kv[2] ** 2) * float(N) ** 3
        k2[0, 0, 0] = 1.0

        def r2c(x):
            h = torch.fft.rfftn(x) / k2
            h[0, 0, 0] = 0
            return h
        h = r2c(g)
        disp = [self.c2r(1j * k * h) for k in kv]
        if order == 2:
            gr = {(a, b): self.c2r(-kv[a] * kv[b] * h) for a in range(3) for b in range(a, 3)}
            src = (gr[0, 0] * gr[1, 1] + gr[0, 0] * gr[2, 2] + gr[1, 1] * gr[2, 2] - gr[0, 1] ** 2 - gr[0, 2] ** 2 -
                   gr[1, 2] ** 2)
            del gr
            s = r2c(src)
            second = [self.c2r(-1j * k * s) for k in kv]
        x = self.axis()
        out = torch.zeros(N ** 3, dtype=torch.float64, device=self.dev)
        for sl in self.chunks():
            r = self.radius(sl)
            D = self.D(r)
            D2 = self.tab("d2", r, None) if order == 2 else None
            cell, wt = [], []
            for ax, x0 in enumerate((x[None, None, :], x[None, :, None], x[sl][:, None, None])):
                q = x0 + 0.5 * self.L + D * disp[ax][sl]
                if order == 2:
                    q = q + D2 * second[ax][sl]
                q = torch.remainder(q, self.L) / self.dx
                if interp == 1:
                    i0 = torch.floor(q).long()
                    f = q - i0
                    cell.append([i0 % N, (i0 + 1) % N])
                    wt.append([1 - f, f])
                else:
                    i0 = torch.floor(q + 0.5).long()
                    f = q - i0
                    cell.append([(i0 + o) % N for o in (-1, 0, 1)])
                    wt.append([0.5 * (0.5 - f) ** 2, 0.75 - f * f, 0.5 * (0.5 + f) ** 2])
            for c2, w2 in zip(cell[2], wt[2]):
                for c1, w1 in zip(cell[1], wt[1]):
                    for c0, w0 in zip(cell[0], wt[0]):
                        out.index_add_(0, (c0 + N * (c1 + N * c2)).reshape(-1), (w0 * w1 * w2).reshape(-1))
        return out.reshape(N, N, N) - 1

    # -- shells ------------------------------------------------------------
    @staticmethod
    def bias(d, b, model):
        if model == 1:
            return torch.where(d < 0, torch.exp(b * d / (1 + d)), 1 + b * d)
        if model == 2:
            return torch.clamp(1 + b * d, min=0)
        return torch.exp(b * torch.log1p(d))

    def shells(self, dens, tracers):
        """[counts, z sums, bias sums, norm tables] of the shells (density.c:1128-1355)."""
        zmax = float(self.z(self.t([0.5 * self.L]))[0])
        nz = int(zmax / 0.05) + 2
        idz = (nz - 2) / zmax
        acc = torch.zeros((2 + len(tracers), nz), dtype=torch.float64, device=self.dev)
        for sl in self.chunks():
            r = self.radius(sl)
            z = self.z(r)
            s = (z * idz).long() + 1
            ok = s < nz
            sv, rv, d = s[ok], r[ok], dens[sl][ok]
            acc[0] += torch.bincount(sv, minlength=nz)
            acc[1] += torch.bincount(sv, weights=z[ok], minlength=nz)
            for t, (_, _, model, _, bz) in enumerate(tracers):
                v = torch.where(d <= -1, torch.zeros_like(d), self.bias(d, self.tab(bz, rv, None, 1.0), model))
                acc[2 + t] += torch.bincount(sv, weights=v, minlength=nz)
        a = acc.cpu().numpy()
        cnt, zs, sums = a[0], a[1], a[2:]
        one = np.maximum(cnt, 1)
        zm = zs / one
        zm[0], zm[-1] = 0, zmax
        ztab = self.z(self.r_arr).cpu().numpy()
        tabs = []
        for sm in sums:
            n = np.where(cnt > 0, cnt / np.where(sm == 0, 1, sm), sm)
            n[0], n[-1] = n[1], n[-2]
            tabs.append(np.interp(ztab, zm, n))
        return [cnt.astype(np.uint64), zs, sums, np.stack(tabs)]

    # -- lines of sight ------------------------------------------------------
    def pix2vec(self, nside):
        """Centres of all NEST pixels (Gorski et al. 2005)."""
        p = torch.arange(12 * nside * nside, device=self.dev)
        face, f = p // (nside * nside), p % (nside * nside)
        ix, iy = torch.zeros_like(f), torch.zeros_like(f)
        for b in range(nside.bit_length()):
            ix |= ((f >> (2 * b)) & 1) << b
            iy |= ((f >> (2 * b + 1)) & 1) << b
        jr = (face // 4 + 2) * nside - ix - iy - 1
        north, south = jr < nside, jr > 3 * nside
        nr = torch.where(north, jr, torch.where(south, 4 * nside - jr, torch.full_like(jr, nside)))
        f2 = 4.0 / (12.0 * nside * nside)
        cap = nr.double() ** 2 * f2
        z = torch.where(north, 1 - cap, torch.where(south, cap - 1, (2 * nside - jr).double() * ((2.0 * nside) * f2)))
        shift = torch.where(north | south, torch.zeros_like(jr), (jr - nside) & 1)
        jpll = torch.tensor([1, 3, 5, 7, 0, 2, 4, 6, 1, 3, 5, 7], device=self.dev)[face]
        jp = torch.div(jpll * nr + ix - iy + 1 + shift, 2, rounding_mode="floor")
        jp = torch.where(jp > 4 * nside, jp - 4 * nside, torch.where(jp < 1, jp + 4 * nside, jp))
        ph = (jp - 0.5 * (shift + 1).double()) * (0.5 * math.pi / nr.double())
        st = torch.sqrt((1 - z) * (1 + z))
        return [st * torch.cos(ph), st * torch.sin(ph), z]

    def tidal(self, phi, i):
        """The six second differences (xx xy xz yy yz zz) of phi at cells i = (x, y, z)."""
        N = self.N
        at = lambda dx, dy, dz: phi[(i[2] + dz) % N, (i[1] + dy) % N, (i[0] + dx) % N]  # noqa: E731
        e = [(1, 0, 0), (0, 1, 0), (0, 0, 1)]
        c0, t = at(0, 0, 0), {}
        for a in range(3):
            t[a, a] = at(*e[a]) + at(*[-v for v in e[a]]) - 2 * c0
            for b in range(a + 1, 3):
                p, m = [x + y for x, y in zip(e[a], e[b])], [x - y for x, y in zip(e[a], e[b])]
                t[a, b] = 0.25 * (at(*p) + at(*[-v for v in p]) - at(*m) - at(*[-v for v in m]))
        return [t[0, 0], t[0, 1], t[0, 2], t[1, 1], t[1, 2], t[2, 2]]

    def central(self, phi, i):
        N = self.N
        at = lambda dx, dy, dz: phi[(i[2] + dz) % N, (i[1] + dy) % N, (i[0] + dx) % N]  # noqa: E731
        return [at(1, 0, 0) - at(-1, 0, 0), at(0, 1, 0) - at(0, -1, 0), at(0, 0, 1) - at(0, 0, -1)]

    def nearest(self, rm, u):
        # the map definition's own expression: rays along rational directions do land on cell edges
        return [((rm * v + 0.5 * self.L) * (self.N / self.L) + 0.5).long() % self.N for v in u]

    def corners(self, x):
        """Cells and weights of the trilinear interpolation at grid coordinates x."""
        i0 = [v.long() for v in x]
        h = [v - i for v, i in zip(x, i0)]
        for c in range(8):
            b = (c & 1, (c >> 1) & 1, c >> 2)
            w = 1.0
            for ax in range(3):
                w = w * (h[ax] if b[ax] else 1 - h[ax])
            yield [(i + o) % self.N for i, o in zip(i0, b)], w

    @staticmethod
    def angles(u):
        cth = u[2].clamp(-1, 1)
        sth = torch.sqrt((1 - cth) * (1 + cth))
        safe = torch.where(sth == 0, torch.ones_like(sth), sth)
        return cth, sth, torch.where(sth == 0, torch.ones_like(sth), u[0] / safe), torch.where(
            sth == 0, torch.zeros_like(sth), u[1] / safe)

    def rotation(self, u):
        cth, sth, cph, sph = self.angles(u)
        return [cth ** 2 * cph ** 2 + sph ** 2, 2 * cph * sph * (cth ** 2 - 1), -2 * cth * sth * cph,
                cth ** 2 * sph ** 2 + cph ** 2, -2 * cth * sth * sph, sth ** 2]

    def los(self, phi, nside, r_src):
        """Convergence and ISW maps (kappa.c:78-175, isw.c:78-147)."""
        u = self.pix2vec(nside)
        rot = [v / self.dx ** 2 for v in self.rotation(u)]
        ih = np.array([int(r / self.dr + 0.5) for r in r_src])
        last = np.minimum(ih, self.nr - 1)
        rm = (torch.arange(self.nr, device=self.dev, dtype=torch.float64) + 0.5) * self.dr
        pg = (self.D(rm) * (1 + self.z(rm))).cpu().numpy()
        pd = self.tab("pd", rm, None).cpu().numpy()
        k1, k2, s = torch.zeros_like(u[0]), torch.zeros_like(u[0]), torch.zeros_like(u[0])
        kap, isw, done = [], [], 0
        for p in range(len(r_src)):
            for j in range(done, last[p] + 1):
                r = (j + 0.5) * self.dr
                i = self.nearest(r, u)
                dot = sum(a * b for a, b in zip(rot, self.tidal(phi, i)))
                k1 += dot * (r * pg[j] * self.dr)
                k2 += dot * (r * r * pg[j] * self.dr)
                s += phi[i[2], i[1], i[0]] * (2 * pd[j] * self.dr)
            done = last[p] + 1
            kap.append(k1 - k2 / (ih[p] * self.dr))
            isw.append(s.clone())
        return torch.stack(kap), torch.stack(isw)

    def custom(self, dens, tracer, table, nside):
        """cstm.c:39-150."""
        _, _, model, amp, bz = tracer
        rm = (torch.arange(self.nr, device=self.dev, dtype=torch.float64) + 0.5) * self.dr
        kz = (self.tab(amp, rm, 0.0, 0.0) / self.tab("ih", rm, None)).cpu().numpy()
        b = self.tab(bz, rm, None, 1.0).cpu().numpy()
        nrm = self.tab(table, rm, None).cpu().numpy()
        on = np.nonzero(np.abs(kz) > 1e-4 * kz.max())[0]
        u = self.pix2vec(nside)
        out = torch.zeros_like(u[0])
        for j in range(on[0], on[-1] + 1):
            d = torch.zeros_like(out)
            for c, w in self.corners([((j + 0.5) * self.dr * v + 0.5 * self.L) / self.dx for v in u]):
                d += dens[c[2], c[1], c[0]] * w
            out += kz[j] * (self.bias(d, float(b[j]), model) * nrm[j] - 1)
        return out * self.dr

    # -- sources -------------------------------------------------------------
    def sample(self, dens, phi, tracer, table, seed):
        """Catalogue (x, y, z, dz) of a population (srcs.c:120-283): counts by
        inversion of the Poisson distribution, one uniform per cell."""
        _, ipop, model, amp, bz = tracer
        N, cell, count = self.N, [], []
        for sl in self.chunks():
            r = self.radius(sl)
            nd = torch.where(r < 0.5 * self.L + 20, self.tab(amp, r, 0.0, 0.0), torch.zeros_like(r))
            d = dens[sl].double()
            lam = nd * self.dx ** 3 * self.bias(d, self.tab(bz, r, None, 1.0), model) * self.tab(table, r, None)
            lam = torch.where((nd > 0) & (d > -1), lam, torch.zeros_like(lam)).reshape(-1)
            base = sl.start * N * N
            w = _philox(torch.arange(base // 8, (base + len(lam)) // 8, device=self.dev), 0, 0x100 + ipop, 0, seed)
            hi = torch.stack([x for v in w for x in (v & 0xFFFF, v >> 16)], dim=1).reshape(-1)
            some = torch.nonzero((hi + 1).double() / 65536 > torch.exp(-lam))[:, 0]
            c, lam, hi = some + base, lam[some], hi[some]
            lo = _philox(c & _M32, c >> 32, 0x40000100 + ipop, 0, seed)[0] & 0xFFFF
            if len(c) == 0:
                continue
            if float(lam.max()) > 500:
                return None
            x = (hi * 65536 + lo).double() / 2.0 ** 32
            p = torch.exp(-lam)
            F, k = p.clone(), torch.zeros_like(c)
            while True:
                more = x > F
                if not bool(more.any()) or int(k.max()) > 6000:
                    break
                k += more
                p = torch.where(more, p * lam / k.clamp(min=1), p)
                F = torch.where(more, F + p, F)
            cell.append(c[k > 0])
            count.append(k[k > 0])
        cell, count = torch.cat(cell), torch.cat(count)
        first = torch.cumsum(count, 0) - count
        c = torch.repeat_interleave(cell, count)
        j = torch.arange(len(c), device=self.dev) - torch.repeat_interleave(first, count)
        i = [c % N, (c // N) % N, c // (N * N)]
        x0 = [v.double() * self.dx - 0.5 * self.L for v in i]
        pos = []
        for ax in range(3):
            n = 3 * j + ax
            w = torch.stack(_philox(c & _M32, c >> 32, 0x200 + ipop, n >> 2, seed))
            u = w.gather(0, (n & 3)[None])[0].double() / 2.0 ** 32
            pos.append(x0[ax] + self.dx * (u - 0.5))
        r = torch.sqrt(x0[0] ** 2 + x0[1] ** 2 + x0[2] ** 2)
        v = sum(a.double() * b for a, b in zip(self.central(phi, i), x0)) / r.clamp(min=1e-30) * (0.5 / self.dx)
        return torch.stack(pos + [v * self.factor_vel() * self.tab("v1", r, None)], dim=1)

    def factor_vel(self):
        return -self.ta["fgrowth_0"] / (1.5 * self.ta["hubble_0"] * self.ta["omega_m"])

    def directions(self, pos):
        p = [pos[:, a].float().double() for a in range(3)]
        r = torch.sqrt(p[0] ** 2 + p[1] ** 2 + p[2] ** 2)
        return p, r, [v / r.clamp(min=0.001) for v in p]

    def velocity(self, phi, x, u):
        v = 0
        for c, w in self.corners(x):
            v = v + w * sum(a * b for a, b in zip(self.central(phi, c), u))
        return v * (0.5 / self.dx)

    def beams(self, phi, pos, a2r):
        """srcs.c:425-737: (dz_rsd, [e1 e2 kappa dra ddec])."""
        p, r, u = self.directions(pos)
        vr = self.velocity(phi, [(v + 0.5 * self.L) / self.dx for v in p], u)
        a = 1 / (1 + self.z(r))
        a2r = self.t(a2r)
        ia = (a * (len(a2r) - 1)).long().clamp(0, len(a2r) - 2)
        rz = torch.where(a >= 1, torch.zeros_like(a), a2r[ia] + (a2r[ia + 1] - a2r[ia]) * (a * (len(a2r) - 1) - ia))
        dz = vr * self.tab("v1", rz, None) * self.factor_vel()
        cth, sth, cph, sph = self.angles(u)
        ir = 1 / r.clamp(min=0.001)
        pre, prem = ir / self.dx ** 2, 0.5 * ir / self.dx
        ux, uy = [cth * cph * prem, cth * sph * prem, -sth * prem], [-sph * prem, cph * prem, torch.zeros_like(r)]
        rk = self.rotation(u)
        re1 = [cth ** 2 * cph ** 2 - sph ** 2, 2 * cph * sph * (cth ** 2 + 1), -2 * cth * sth * cph,
               cth ** 2 * sph ** 2 - cph ** 2, -2 * cth * sth * sph, sth ** 2]
        re2 = [-2 * cth * cph * sph, 2 * cth * (cph ** 2 - sph ** 2), 2 * sth * sph, 2 * cth * sph * cph,
               -2 * sth * cph, torch.zeros_like(r)]
        o = [torch.zeros_like(r) for _ in range(5)]
        last = (r / self.dr + 0.5).long().clamp(max=self.nr - 1)
        rm = (torch.arange(self.nr, device=self.dev, dtype=torch.float64) + 0.5) * self.dr
        pg = (self.D(rm) * (1 + self.z(rm)) * self.dr).cpu().numpy()
        for j in range(int(last.max()) + 1):
            rj = (j + 0.5) * self.dr
            i = self.nearest(rj, u)
            fr = torch.where(j <= last, rj * pg[j] * (r - rj), torch.zeros_like(r))
            fm = torch.where(j <= last, 2 * pg[j] * (r - rj), torch.zeros_like(r))
            t, v = self.tidal(phi, i), self.central(phi, i)
            for q, m in enumerate((re1, re2, rk)):
                o[q] += fr * pre * sum(x * y for x, y in zip(m, t))
            o[3] += fm * sum(x * y for x, y in zip(uy, v)) * 57.2957795
            o[4] += fm * sum(x * y for x, y in zip(ux, v)) * 57.2957795
        return dz, torch.stack(o, dim=1)

    def skewers(self, dens, phi, pos, gaussian, sigma2):
        """srcs.c:507-529, 725-733."""
        _, r, u = self.directions(pos)
        last = (r / self.dr + 0.5).long().clamp(max=self.nr - 1)
        f = dens
        if gaussian:
            f = torch.empty_like(dens)
            for sl in self.chunks():
                D = self.D(self.radius(sl))
                f[sl] = torch.log1p(dens[sl]) / D + 0.5 * D * sigma2
        dg = torch.zeros((len(r), self.nr), dtype=torch.float64, device=self.dev)
        vs = torch.zeros_like(dg)
        rm = (torch.arange(self.nr, device=self.dev, dtype=torch.float64) + 0.5) * self.dr
        v1 = self.tab("v1", rm, None).cpu().numpy() * self.factor_vel()
        for j in range(self.nr):
            x = [((j + 0.5) * self.dr * v + 0.5 * self.L) / self.dx for v in u]
            d = sum(w * f[c[2], c[1], c[0]] for c, w in self.corners(x))
            on = (j <= last).double()
            dg[:, j] = d * on
            vs[:, j] = self.velocity(phi, x, u) * v1[j] * on
        return dg, vs

    # -- intensity maps ------------------------------------------------------
    def ang2pix(self, nside, cth, phi):
        """RING pixel of a direction (Gorski et al. 2005)."""
        tt = phi * (2 / math.pi)
        t1, t2 = nside * (0.5 + tt), nside * cth * 0.75
        jp, jm = (t1 - t2).long(), (t1 + t2).long()
        ir = nside + 1 + jp - jm
        ip = torch.div(jp + jm - nside + (1 - (ir & 1)) + 1, 2, rounding_mode="floor") % (4 * nside)
        eq = nside * (nside - 1) * 2 + (ir - 1) * 4 * nside + ip
        tp = tt - tt.long()
        tmp = nside * torch.sqrt(3 * (1 - cth.abs()))
        ir = (tp * tmp).long() + ((1 - tp) * tmp).long() + 1
        ip = (tt * ir).long() % (4 * ir)
        cap = torch.where(cth > 0, 2 * ir * (ir - 1) + ip, 12 * nside * nside - 2 * ir * (ir + 1) + ip)
        return torch.where(cth.abs() <= 2.0 / 3.0, eq, cap)

    def imap(self, dens, phi, tracer, table, nside, r0, rf):
        """imap.c:135-245 for contiguous shells: (temperature, hit count) sums."""
        _, _, model, amp, bz = tracer
        o = np.argsort(r0)
        r0, rf = r0[o], rf[o]
        npix, nr = 12 * nside * nside, len(r0)
        edges = self.t(np.append(r0, rf[-1]))
        size = math.sqrt(4 * math.pi / npix)
        sc = np.minimum(np.minimum(((rf ** 3 - r0 ** 3) * size * size / 3) ** 0.333333, r0 * size), rf - r0)
        nsub = torch.as_tensor((self.dx / sc + 0.5).astype(np.int64) + 1, device=self.dev)
        data = torch.zeros(nr * npix, dtype=torch.float64, device=self.dev)
        nadd = torch.zeros(nr * npix, dtype=torch.int64, device=self.dev)
        x = self.axis()
        for sl in self.chunks():
            r = self.radius(sl)
            T = self.tab(amp, r, 0.0, 0.0)
            k, y, xx = torch.nonzero((r <= rf[-1] + 20) & (r >= r0[0] - 20) & (T > 0), as_tuple=True)
            i = [xx, y, k + sl.start]
            rr, d = r[k, y, xx], dens[i[2], i[1], i[0]].double()
            T = T[k, y, xx] * self.bias(d, self.tab(bz, rr, None, 1.0), model) * self.tab(table, rr, None)
            c = [x[v] for v in i]
            v = sum(a.double() * b for a, b in zip(self.central(phi, i), c)) / rr.clamp(min=1e-30) * (0.5 / self.dx)
            shift = v * self.factor_vel() * self.tab("v1", rr, None) * self.tab("ih", rr, None)
            shift = torch.where(rr > 0, shift, torch.zeros_like(shift))
            ns_cell = nsub[(torch.bucketize(rr, edges, right=True) - 1).clamp(0, nr - 1)]
            for ns in torch.unique(ns_cell).tolist():
                m = ns_cell == ns
                cm, Tm, sm = [a[m] for a in c], T[m], shift[m]
                off = torch.arange(ns ** 3, device=self.dev)
                step = max(1, (1 << 24) // max(1, len(Tm)))
                for a in range(0, ns ** 3, step):
                    oo = off[a:a + step]
                    q = [cm[ax][:, None] + ((oo // ns ** ax) % ns + 0.5).double()[None, :] * (self.dx / ns) for ax in range(3)]
                    rq = torch.sqrt(q[0] ** 2 + q[1] ** 2 + q[2] ** 2)
                    ish = torch.bucketize(rq + sm[:, None], edges, right=True) - 1
                    ok = (ish >= 0) & (ish < nr)
                    ph = torch.atan2(q[1] / rq, q[0] / rq)
                    ph = torch.where(ph < 0, ph + 2 * math.pi, ph)
                    pix = (ish * npix + self.ang2pix(nside, q[2] / rq, ph))[ok]
                    data.index_add_(0, pix, Tm[:, None].expand(-1, len(oo))[ok])
                    nadd += torch.bincount(pix, minlength=nr * npix)
        # rows in the caller's shell order are rows of the sorted shells
        return data.reshape(nr, npix), nadd.reshape(nr, npix).int()


def exact(case, seed):
    e = _Exact(case)
    kind, run, seed32 = case["kind"], e.run, _seed32(seed)
    tracers = _tracers(case, run)
    rs = run.scalar("r_smooth")
    if kind in ("chain", "maps", "lpt"):
        dens, phi = e.fields(seed32, rs, case.get("smooth_potential", True))
        s2 = float(dens.var(correction=0))
        if kind == "lpt":
            del phi
            dens = e.lpt(dens, case["order"], case["interp"])
        else:
            dens = e.density(dens, s2, case.get("density_type") == "clip")
        norms = e.shells(dens, tracers)
        out = dict(sigma2=s2, norms=norms)
        if kind != "lpt":
            r_src = _planes(run, case["z_max"])
            kap, isw = e.los(phi, case["nside"], r_src[-1:] if kind == "chain" else r_src)
            out["kappa"] = kap
        if kind == "chain":
            # a source more or less moves every later row: the catalogues have no counterpart from other fields
            out["catalogues"] = None
        elif kind == "maps":
            out["isw"] = isw
        if kind == "lpt" or case.get("custom"):
            out["custom"] = e.custom(dens, tracers[-1], norms[3][-1], case["nside"])
        return out
    dens, phi, s2 = _gaussian_grid(case, run, seed)
    tables = e.shells(dens.double(), tracers)[3]
    if kind == "imap":
        nside, r0, rf = run.imap_shells(0)
        return list(e.imap(dens, phi, tracers[0], tables[0], nside, r0, rf))
    cats = [e.sample(dens, phi, t, tab, seed32) for t, tab in zip(tracers, tables)]
    if any(c is None for c in cats):
        return None
    caps = [max(len(c), _capacity(run, t[3])) for c, t in zip(cats, tracers)]
    pad = lambda v, cap: torch.nn.functional.pad(v, [0, 0] * (v.dim() - 1) + [0, cap - len(v)])  # noqa: E731
    if kind == "sources":
        return [(len(c), pad(c, cap), None) for c, cap in zip(cats, caps)]
    if kind == "beams":
        return [pad(v, caps[0]) for v in e.beams(phi.double(), cats[0], run.r_a2r())]
    return [pad(v, caps[0]) for v in e.skewers(dens.double(), phi.double(), cats[0], case["gaussian"], s2)]
