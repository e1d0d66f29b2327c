"""Count bytes of blocks without sources.

k_count sets the bytes of a 512-cell block only where one is not 0, and k_fill
and the count fetch read only blocks that hold sources.  On one context a dense
call (escaped counts, every block full) is followed by sparser ones whose empty
blocks still hold its bytes: catalogue, cell counts and their sum against the
oracle at each density, at grids whose blocks span several rows and parts of rows.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,scales", [
    (32, (1.0, 1e-2, 1e-4, 3e-6)),
    (64, (1.0, 1e-3, 1e-5, 1e-2)),
    (192, (0.3, 1e-4, 1e-6)),   # the most blocks of the one-kernel scan
    (256, (1e-2, 1e-6)),        # three scan kernels
])
def test_dense_then_sparse(workdir, N, scales):
    from colore_amd import lib
    from oracle_lib import Oracle
    _, run = make_run("C1", N, workdir, with_maps=False)
    L = run.scalar("l_box")
    ctx = lib.Context(N, L)
    ctx.upload_tables(run.tables())
    orc = Oracle(run.table_arrays())
    amp, bz, model = run.tracer(0, 0)
    s2 = ctx.gaussian_fields(77, run.scalar("r_smooth"), True)
    ctx.set_tracer(0, 0, model, amp, bz)
    ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
    dens = ctx.fetch_grid(0).astype(np.float64)
    npot = ctx.fetch_grid(1).astype(np.float64)
    tab, n0, nf = ctx.norm_table(0, 0)
    top = 0
    for s in scales:
        ctx.set_tracer(0, 0, model, amp * s, bz)
        ctx.set_norm_table(0, 0, tab, n0, nf)
        n = ctx.sample_sources(0, 77, 2)
        pop = orc.pop(N, L, amp * s, bz, tab, n0, nf, model, 0, 77)
        tot, counts = orc.counts(pop, dens)
        assert n == tot
        got = ctx.fetch_cell_counts(0, 0, N)
        assert np.array_equal(got.reshape(-1), np.asarray(counts).reshape(-1))
        top = max(top, got.max())
        if n:
            pos, ipix = ctx.fetch_sources(0, n)
            opos, oipix = orc.sources(pop, dens, npot, 2, cap=n + 1)
            assert np.array_equal(pos[:, :3], opos[:, :3]) and np.array_equal(ipix, oipix)
    assert N != 32 or top > 255
    ctx.close()
