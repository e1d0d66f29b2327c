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
