"""Line-of-sight marches over the forms their kernels split into.

kappa, ISW and custom maps march with 1 to 16 lanes per pixel (by map size and
steps) and kappa with per-cell records or straight from the potential (by
steps per cell).  Every combination is compared with the FP64 oracle on the
same grids (1e-5 of the map RMS, as in test_los_maps), with one and several
source planes, two of them equal, and for an observer off the box's centre,
whose rays wrap around the box.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nside,off", [
    (32, 1, 0.0),      # 12 pixels, the fewest steps
    (64, 8, 0.0),      # several lanes per pixel, direct
    (64, 64, 0.11),    # records
    (128, 16, 0.23),   # direct, wrapping
    (128, 128, 0.23),  # records, wrapping, one lane per pixel
    (192, 32, 0.0),
])
def test_maps_vs_oracle(workdir, N, nside, off):
    from colore_amd import lib
    from oracle_lib import Oracle
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    L, rmax = run.scalar("l_box"), run.scalar("r_max")
    obs = np.array([0.5 + off, 0.5 - off, 0.5 + 0.5 * off]) * L
    ctx = lib.Context(N, L, pos_obs=obs)
    ctx.upload_tables(run.tables())
    ctx.gaussian_fields(5, 2.0, True)
    phi = ctx.fetch_grid(1).astype(np.float64)
    orc = Oracle(run.table_arrays())
    for planes in ([rmax], [0.3 * rmax, 0.8 * rmax, 0.8 * rmax, rmax]):
        r = np.array(planes)
        for which, got in ((0, ctx.kappa(nside, r)), (1, ctx.isw(nside, r))):
            want = _oracle_maps(orc, which, N, L, obs, rmax, phi, nside, r)
            rms = np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))
            assert (np.abs(got - want) / rms).max() < 1e-5, (which, planes)
    ctx.close()


def _oracle_maps(orc, which, N, L, obs, rmax, phi, nside, r):
    import ctypes
    from oracle_lib import p
    out = np.zeros((len(r), 12 * nside * nside))
    g = np.ascontiguousarray(phi)
    orc.lib.orc_kappa_isw(which, N, L, p(np.ascontiguousarray(obs)), rmax, ctypes.byref(orc.bg), p(g), nside, len(r),
                          p(np.ascontiguousarray(r)), p(out))
    return out


@pytest.mark.parametrize("N,nside,off,lo,hi", [
    (64, 256, 0.11, 0.0, 1.0),     # one lane per pixel, wrapping
    (128, 128, 0.23, 0.1, 0.93),   # 2 lanes per pixel, 54 steps
    (64, 16, 0.0, 0.0, 1.0),       # 4
    (128, 8, 0.11, 0.0, 1.0),      # 8
    (256, 8, 0.23, 0.0, 0.99),     # 8, 127 steps
    (256, 8, 0.0, 0.0, 1.0),       # 16
    (64, 16, 0.23, 0.48, 0.51),    # a single step
    (64, 16, 0.11, 0.3, 0.75),     # 14 steps: one lane for a small map
])
def test_custom_maps_vs_oracle(workdir, N, nside, off, lo, hi):
    """Kernels K(r) of 1 between lo and hi of r_max, every bias model."""
    import ctypes
    from colore_amd import lib
    from oracle_lib import Oracle, p
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    L, rmax = run.scalar("l_box"), run.scalar("r_max")
    obs = np.array([0.5 + off, 0.5 - off, 0.5 + 0.5 * off]) * L
    ctx = lib.Context(N, L, pos_obs=obs)
    ctx.upload_tables(run.tables())
    s2 = ctx.gaussian_fields(5, 2.0, True)
    ctx.density(lib.CLR_DENS_LOGNORMAL, s2)
    dens = ctx.fetch_grid(0).astype(np.float64)
    orc = Oracle(run.table_arrays())
    r = run.table_arrays()["r"]
    kz = ((r >= lo * rmax) & (r <= hi * rmax)).astype(np.float64)
    norm = 1.0 + 0.1 * r / rmax
    for model, b in ((lib.CLR_BIAS_EXPONENTIAL, 1.3), (lib.CLR_BIAS_EXP_TRUNCATED, 1.5), (lib.CLR_BIAS_TRUNCATED, 2.2)):
        bz = b * (1 + 0.2 * r / rmax)
        ctx.set_tracer(lib.CLR_TRACER_CSTM, 0, model, kz, bz)
        ctx.set_norm_table(lib.CLR_TRACER_CSTM, 0, norm, norm[0], norm[-1])
        got = ctx.custom_map(0, nside)
        want = np.zeros(12 * nside * nside)
        assert orc.lib.orc_cstm(N, L, p(obs), rmax, ctypes.byref(orc.bg), p(dens), p(kz), p(bz), p(norm), norm[0],
                                norm[-1], model, nside, p(want)) == 0
        rms = np.sqrt(np.mean(want ** 2))
        assert rms > 0
        assert np.abs(got - want).max() <= 1e-5 * rms, model
    ctx.close()
