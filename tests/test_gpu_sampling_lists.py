"""Sampling calls whose lists outgrow their first sizes.

With 400 sources in every cell of 64^3 all counts go through the FP64 queue and
end in the escape list, and both lists overflow their 65536 entries; how long the
second one must be is only known once the first is long enough.  Cell counts
equal to the oracle's.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


def test_both_lists_overflow(workdir):
    from colore_amd import lib
    from oracle_lib import Oracle
    N = 64
    _, run = make_run("C1", N, workdir, with_maps=False)
    L = run.scalar("l_box")
    ctx = lib.Context(N, L)
    ctx.upload_tables(run.tables())
    amp, bz, model = run.tracer(0, 0)
    s2 = ctx.gaussian_fields(77, run.scalar("r_smooth"), True)
    ctx.set_tracer(0, 0, model, amp, bz)
    ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
    dens = ctx.fetch_grid(0).astype(np.float64)
    tab, n0, nf = ctx.norm_table(0, 0)
    amp = np.full_like(amp, 400 / (L / N) ** 3)
    ctx.set_tracer(0, 0, model, amp, bz)
    ctx.set_norm_table(0, 0, tab, n0, nf)
    n = ctx.sample_sources(0, 77, 2)
    got = ctx.fetch_cell_counts(0, 0, N)
    orc = Oracle(run.table_arrays())
    tot, counts = orc.counts(orc.pop(N, L, amp, bz, tab, n0, nf, model, 0, 77), dens)
    assert (counts >= 254).sum() > 65536
    assert n == tot and np.array_equal(got.reshape(-1), np.asarray(counts).reshape(-1))
    # the lists have their sizes now
    assert ctx.sample_sources(0, 77, 2) == n
    ctx.close()
