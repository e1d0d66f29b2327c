"""Source planes at distances that take no step: negative, NaN, past any grid.

Such a plane's map holds nothing of the field, and the planes sorted after it
are those of a call without it (also those after a distance that rounds to step
0, whose own map divides by 0 as in the reference).
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nside", [(64, 4), (64, 64), (128, 128)])   # several lanes per pixel, records, one lane
def test_planes_without_steps(workdir, N, nside):
    from colore_amd import lib
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    rmax = run.scalar("r_max")
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    ctx.gaussian_fields(5, 2.0, True)
    good = [0.4 * rmax, 0.9 * rmax]
    for call in (ctx.kappa, ctx.isw):
        want = call(nside, np.array(good))
        assert np.abs(want).max() > 0
        for bad in ([-0.3 * rmax], [-1e12], [np.nan], [-np.inf, -2.5 * rmax / N], [-5 * rmax, np.nan]):
            got = call(nside, np.array(good + bad))
            assert np.array_equal(got[len(bad):], want), bad
            for m, d in zip(got, sorted(bad, key=lambda d: -np.inf if np.isnan(d) else d)):
                if not d / (2 * rmax / N) + 0.5 > -1:
                    assert not m.any(), (bad, d)
        for far in (1e300, np.inf):
            assert np.array_equal(call(nside, np.array([far] + good))[:2], want), far
    ctx.close()


@pytest.mark.parametrize("N,nside,nplanes", [
    (32, 1, 100), (32, 64, 30),    # more planes than steps
    (64, 4, 10), (64, 4, 100),     # direct, several lanes per pixel
    (64, 64, 4), (128, 64, 37),    # records
    (128, 128, 12),                # one lane per pixel
])
def test_many_planes_vs_oracle(workdir, N, nside, nplanes):
    """Planes that end within a few steps of each other, some at the same step:
    every plane within 1e-5 of its RMS (as in test_maps_vs_oracle)."""
    from colore_amd import lib
    from oracle_lib import Oracle
    from test_gpu_march import _oracle_maps
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    L, rmax = run.scalar("l_box"), run.scalar("r_max")
    obs = np.array([0.55, 0.45, 0.525]) * L
    ctx = lib.Context(N, L, pos_obs=obs)
    ctx.upload_tables(run.tables())
    ctx.gaussian_fields(5, 2.0, True)
    phi = ctx.fetch_grid(1).astype(np.float64)
    orc = Oracle(run.table_arrays())
    r = np.linspace(0.1, 1, nplanes) * rmax
    for which, got in ((0, ctx.kappa(nside, r)), (1, ctx.isw(nside, r))):
        want = _oracle_maps(orc, which, N, L, obs, rmax, phi, nside, r)
        rms = np.sqrt(np.mean(want ** 2, axis=1, keepdims=True))
        assert (np.abs(got - want) / rms).max() < 1e-5, which
    ctx.close()


def test_planes_a_float_apart(workdir):
    """Two distances that are one float on both sides of a rounding step: planes
    are sorted by their float values, so the farther one may come first.  The
    planes of three and of more than three planes' march are the same."""
    from colore_amd import lib
    N = 64
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    rmax = run.scalar("r_max")
    tie = 10.5 * 2 * rmax / N
    near = [tie * (1 + 1e-9), tie * (1 - 1e-9), 0.7 * rmax]
    assert len({np.float32(d) for d in near[:2]}) == 1
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    ctx.gaussian_fields(5, 2.0, True)
    for nside in (1, 64):
        for call in (ctx.kappa, ctx.isw):
            want = call(nside, np.array(near))
            got = call(nside, np.array(near + list(np.linspace(0.8, 1, 8) * rmax)))
            assert np.array_equal(got[:3], want)
    ctx.close()
