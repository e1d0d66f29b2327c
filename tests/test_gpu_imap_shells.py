"""21cm maps whose cells reach several shells.

Cells that reach at most two shells find a sub-point's by one comparison, the
others by a search; both take the shortened pixel where it is certain.  Hit
counts equal to the oracle's (the sums of the same sub-points are compared in
test_imap_vs_oracle).
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nside,bands", [(32, 16, 40), (64, 16, 64), (64, 64, 24), (128, 8, 3)])
def test_hit_counts(workdir, N, nside, bands):
    from colore_amd import lib
    from oracle_lib import Oracle
    _, run = make_run("C3", N, workdir, z_max=1.5, imap_bands=bands, imap_nside=nside)
    L = run.scalar("l_box")
    ctx = lib.Context(N, L)
    ctx.upload_tables(run.tables())
    tz, bz, model = run.tracer(1, 0)
    ctx.set_tracer(1, 0, model, tz, bz)
    s2 = ctx.gaussian_fields(3003, run.scalar("r_smooth"), True)
    ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
    dens, npot = (ctx.fetch_grid(k).astype(np.float64) for k in (0, 1))
    nside, r0, rf = run.imap_shells(0)
    tab, n0, nf = ctx.norm_table(1, 0)
    _, nadd = ctx.imap(0, nside, r0, rf)
    ctx.close()
    _, want = Oracle(run.table_arrays()).imap(N, L, dens, npot, tz, bz, tab, n0, nf, model, nside, r0, rf)
    assert want.sum() > 0
    assert np.array_equal(nadd, want)
