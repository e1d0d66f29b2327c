"""The sources' line-of-sight pass and skewers in order of direction.

Large catalogues on large grids are marched in the order of the sources'
directions, small ones with several lanes per source: both sides of each line.
2000 sources of each catalogue against the FP64 oracle, every value within
1e-5 of its column's RMS (as in test_source_beams).
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


def _sampled(run, N, n_want):
    """A context with about n_want sources of the first population."""
    from colore_amd import lib
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    amp, bz, model = run.tracer(0, 0)

    def sample(scale):
        ctx.set_tracer(0, 0, model, amp * scale, bz)
        s2 = ctx.gaussian_fields(11, run.scalar("r_smooth"), True)
        ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
        return ctx.sample_sources(0, 11, 2), s2

    f = 1e-2
    f *= n_want / sample(f)[0]
    n, s2 = sample(f)
    assert abs(n - n_want) < 0.03 * n_want
    return ctx, n, s2


@pytest.mark.parametrize("N,n_want,gaussian", [
    (256, 23000, False),   # just below the order's line
    (256, 26000, False),   # just above it
    (384, 30000, True),
])
def test_skewers_vs_oracle(workdir, N, n_want, gaussian):
    from oracle_lib import Oracle
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False)
    ctx, n, s2 = _sampled(run, N, n_want)
    pos, _ = ctx.fetch_sources(0, n)
    dens, phi = (ctx.fetch_grid(k).astype(np.float64) for k in (0, 1))
    dg, vs = ctx.source_skewers(0, n, gaussian, s2)
    pick = np.concatenate([[0, n - 1], np.random.default_rng(1).choice(n, 998, replace=False)])
    odg, ovs = Oracle(run.table_arrays()).src_skewers(N, run.scalar("l_box"), dens, phi, pos[pick], gaussian, s2)
    for g, o in ((dg[pick], odg), (vs[pick], ovs)):
        rms = np.sqrt(np.mean(o * o))
        assert rms > 0
        assert np.abs(g.astype(np.float64) - o).max() <= 1e-5 * rms
        assert np.array_equal(g == 0, o == 0)
    ctx.close()


@pytest.mark.parametrize("N,n_want", [
    (256, 32000),     # just below the order's line, 8 lanes per source
    (256, 34000),     # just above it
    (256, 300000),    # ordered, one lane per source
    (128, 300000),    # catalogue order, one lane per source
    (64, 3000),       # catalogue order, few steps
])
def test_beams_vs_oracle(workdir, N, n_want):
    from oracle_lib import Oracle
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False)
    L = run.scalar("l_box")
    ctx, n, _ = _sampled(run, N, n_want)
    pos, _ = ctx.fetch_sources(0, n)
    phi = ctx.fetch_grid(1).astype(np.float64)
    dz, lens = ctx.source_beams(0, n, run.r_a2r(), True)
    dz0, _ = ctx.source_beams(0, n, run.r_a2r(), False)
    assert np.array_equal(dz, dz0)
    pick = np.concatenate([[0, n - 1], np.random.default_rng(1).choice(n, min(n, 1998), replace=False)])
    odz, olens = Oracle(run.table_arrays()).src_beams(N, L, phi, pos[pick], run.r_a2r(), True)
    for k, (g, o) in enumerate([(dz[pick], odz)] + [(lens[pick, j], olens[:, j]) for j in range(5)]):
        rms = np.sqrt(np.mean(o * o))
        assert rms > 0, k
        assert np.abs(g.astype(np.float64) - o).max() <= 1e-5 * rms, k
    ctx.close()
