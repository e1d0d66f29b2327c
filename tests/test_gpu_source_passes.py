"""The sources' line-of-sight pass and skewers where their staging splits.

Skewers of more sources than one launch stages, beams of more sources than the
context keeps a buffer for, the march in catalogue order where the order's
scratch does not fit, and observers off the box's centre.  1000 sources of each
against the FP64 oracle, every value within 1e-5 of its column's RMS (as in
test_source_beams).
"""
import ctypes

import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


def _sampled(run, N, n_want, obs=None):
    """A context with about n_want sources of the first population."""
    from colore_amd import lib
    ctx = lib.Context(N, run.scalar("l_box"), pos_obs=obs)
    ctx.upload_tables(run.tables())
    amp, bz, model = run.tracer(0, 0)
    ctx.set_tracer(0, 0, model, amp, bz)
    s2 = ctx.gaussian_fields(11, run.scalar("r_smooth"), True)
    ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
    tab = ctx.norm_table(0, 0)

    def sample(f):
        ctx.set_tracer(0, 0, model, amp * f, bz)
        ctx.set_norm_table(0, 0, *tab)
        return ctx.sample_sources(0, 11, 2)

    f = 1e-3
    n = sample(f * n_want / sample(f))
    assert abs(n - n_want) < 0.05 * n_want
    return ctx, n, s2


def _oracle_beams(run, N, obs, phi, pos):
    from oracle_lib import Oracle, p
    o = Oracle(run.table_arrays())
    t, n, L = o.ta, len(pos), run.scalar("l_box")
    dz, lens = np.zeros(n), np.zeros((n, 5))
    pos = np.ascontiguousarray(pos, dtype=np.float32)
    a2r = np.ascontiguousarray(run.r_a2r(), dtype=np.float64)
    o.lib.orc_src_beams(N, L, p(obs), t["r_max"], ctypes.byref(o.bg), p(a2r), t["fgrowth_0"], t["hubble_0"],
                        t["omega_m"], p(phi), n, p(pos, ctypes.c_float), p(dz), p(lens))
    return dz, lens


def _oracle_skewers(run, N, obs, dens, phi, pos):
    from oracle_lib import Oracle, p
    o = Oracle(run.table_arrays())
    t, n, L = o.ta, len(pos), run.scalar("l_box")
    dg, vs = np.zeros((n, N // 2)), np.zeros((n, N // 2))
    pos = np.ascontiguousarray(pos, dtype=np.float32)
    o.lib.orc_src_skewers(N, L, p(obs), t["r_max"], ctypes.byref(o.bg), t["fgrowth_0"], t["hubble_0"], t["omega_m"],
                          p(dens), p(phi), 0, 0.0, n, p(pos, ctypes.c_float), p(dg), p(vs))
    return dg, vs


def _near(got, want, what):
    rms = np.sqrt(np.mean(want * want))
    assert rms > 0, what
    assert np.abs(got.astype(np.float64) - want).max() <= 1e-5 * rms, what


def _pick(n, m=1000, more=()):
    return np.concatenate([[0, n - 1], np.random.default_rng(1).choice(n, m - 2 - len(more), replace=False),
                           np.asarray(more, dtype=np.int64)])


def _check_beams(run, ctx, N, obs, n, pick):
    phi = ctx.fetch_grid(1).astype(np.float64)
    pos, _ = ctx.fetch_sources(0, n)
    dz, lens = ctx.source_beams(0, n, run.r_a2r(), True)
    odz, olens = _oracle_beams(run, N, obs, phi, pos[pick])
    _near(dz[pick], odz, "dz")
    for k in range(5):
        _near(lens[pick, k], olens[:, k], k)
    return dz, lens


def test_skewers_in_several_launches(workdir):
    """384^3, 2^26 / 192 = 349525 sources per launch: a full one and a smaller one."""
    N, n_want = 384, 400_000
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False)
    obs = np.full(3, 0.5 * run.scalar("l_box"))
    ctx, n, _ = _sampled(run, N, n_want)
    per = (1 << 26) // (N // 2)
    assert per < n < 2 * per
    dens, phi = (ctx.fetch_grid(k).astype(np.float64) for k in (0, 1))
    pos, _ = ctx.fetch_sources(0, n)
    dg, vs = ctx.source_skewers(0, n, False)
    ctx.close()
    pick = _pick(n, more=[per - 1, per, per + 1])
    odg, ovs = _oracle_skewers(run, N, obs, dens, phi, pos[pick])
    _near(dg[pick], odg, "density")
    _near(vs[pick], ovs, "velocity")
    assert np.array_equal(dg[pick] == 0, odg == 0)


def test_beams_beyond_the_kept_buffer(workdir):
    """3.1e7 sources need 36 bytes each, more than the GiB that a context keeps;
    with 0.9 GB of the device free they are marched in catalogue order."""
    from device_memory import free_bytes, only
    N, n_want = 256, 31_000_000
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False)
    obs = np.full(3, 0.5 * run.scalar("l_box"))
    ctx, n, _ = _sampled(run, N, n_want)
    assert 36 * n > 1 << 30
    room = 900_000_000
    assert 24 * n + (1 << 20) < room < 36 * n
    with only(room, slack=1 << 25):
        assert 24 * n < free_bytes() < 36 * n
        before = ctx.lib.clr_device_bytes(ctx.h)
        dz1, lens1 = ctx.source_beams(0, n, run.r_a2r(), True)
        # the buffer without the order's scratch
        assert 24 * n <= ctx.lib.clr_device_bytes(ctx.h) - before < 36 * n
    dz, lens = _check_beams(run, ctx, N, obs, n, _pick(n))
    ctx.close()
    assert np.array_equal(dz, dz1)
    for k in range(5):   # the march straight from the potential instead of the records
        rms = np.sqrt(np.mean(lens[:, k].astype(np.float64) ** 2))
        assert np.abs(lens[:, k] - lens1[:, k]).max() <= 1e-6 * rms, k


@pytest.mark.parametrize("N,n_want,off", [
    (64, 3000, 0.11),      # several lanes per source
    (256, 40000, 0.23),    # in order of direction
    (128, 300000, 0.4),    # one lane per source, an observer near a corner
])
def test_observer_off_centre(workdir, N, n_want, off):
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    obs = np.array([0.5 + off, 0.5 - off, 0.5 + 0.5 * off]) * run.scalar("l_box")
    ctx, n, _ = _sampled(run, N, n_want, obs=obs)
    pick = _pick(n)
    _check_beams(run, ctx, N, obs, n, pick)
    dens, phi = (ctx.fetch_grid(k).astype(np.float64) for k in (0, 1))
    pos, _ = ctx.fetch_sources(0, n)
    dg, vs = ctx.source_skewers(0, n, False)
    ctx.close()
    odg, ovs = _oracle_skewers(run, N, obs, dens, phi, pos[pick])
    _near(dg[pick], odg, "density")
    _near(vs[pick], ovs, "velocity")
