"""The fused count pass works on the float that the shell pass stores.

clr_sample_sources_surrogate applies the lognormal transform per cell where
clr_shell_norms(lognormal_fused) stores it; with equal norm tables the counts
of both must be equal.  The growth table falls by 2^24 across the box, so that
one rounding of a cell's table position is a relative 1e-6 of its mean, and the
grid holds D(r) delta_G of about 2 everywhere with 30 sources per cell: were the
passes to round that position differently, a cell in 1e5 would count one
source more or less.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [64, 128])
def test_fused_counts_steep_growth(workdir, N):
    from colore_amd import lib
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False)
    L = run.scalar("l_box")
    ta = run.table_arrays()
    r_edge = 0.5 * 3 ** 0.5 * L
    ta["d1"] = 0.5 ** (24 * ta["r"] / r_edge)
    ctx = lib.Context(N, L)
    ctx.upload_table_arrays(ta)
    x = (np.arange(N) * (L / N) - 0.5 * L) ** 2
    r = np.sqrt(x[:, None, None] + x[None, :, None] + x[None, None, :])
    g = np.zeros(ctx.padded_shape, dtype=np.float32)
    g[:, :, :N] = np.random.default_rng(3).normal(2.0, 0.3, (N, N, N)) * 2.0 ** (24 * r / r_edge)
    b = np.full(len(ta["r"]), 2.0)
    dx3 = (L / N) ** 3
    amp = np.full(len(ta["r"]), 1e-6 / dx3)

    def fused():
        ctx.set_tracer(0, 0, lib.CLR_BIAS_EXPONENTIAL, amp, b)
        ctx.upload_grid(lib.CLR_GRID_DENS, g)
        ctx.declare_grids(0.0, False)
        n = ctx.sample_sources_surrogate(None, 0, 9, 2)
        return n, ctx.norm_table(0, 0)

    # the population that has 30 sources per cell under the closure's norms
    _, (tab, _, _) = fused()
    amp = 30.0 / (dx3 * tab * np.exp(2.0 * 2.0))
    n, (tab, n0, nf) = fused()
    counts = ctx.fetch_cell_counts(0, 0, N)
    assert n > 10 * N ** 3

    ctx.upload_grid(lib.CLR_GRID_DENS, g)
    ctx.declare_grids(0.0, False)
    ctx.shell_norms(lognormal_fused=True, sigma2=0.0, ntracers=1)
    ctx.set_norm_table(0, 0, tab, n0, nf)
    n2 = ctx.sample_sources(0, 9, 2)
    two = ctx.fetch_cell_counts(0, 0, N)
    ctx.close()
    differ = int((two != counts).sum())
    assert differ == 0 and n2 == n
