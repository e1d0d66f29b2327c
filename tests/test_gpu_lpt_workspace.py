"""LPT densities on a context that keeps its workspace between calls.

Orders, assignment kernels and grid sizes follow each other on one context
(the workspace grows, is reused and holds other data by then), and every
density must equal the one a fresh context computes (deposits add in FP64 or
FP32 in an order that varies: 2e-6 of 1 + delta) with the same mass.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


def _ctx(run, N):
    from colore_amd import lib
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    return ctx


def _density(ctx, seed, order, interp, positions):
    ctx.gaussian_fields(seed, 2.0, True)
    pos = ctx.lpt_density(interp, order, positions=positions)
    return ctx.fetch_grid(0)[:, :, :ctx.N].astype(np.float64), pos


@pytest.mark.parametrize("N", [32, 64, 192, 256])
def test_lpt_calls_in_turn(workdir, N):
    _, run = make_run("C2", N, workdir, z_max=0.6, with_maps=False)
    ctx = _ctx(run, N)
    for seed, order, interp, positions in ((1, 1, 1, False), (2, 2, 2, False), (3, 1, 2, True), (4, 2, 1, True),
                                           (5, 1, 0, False), (6, 1, 1, False)):
        got, gpos = _density(ctx, seed, order, interp, positions)
        fresh = _ctx(run, N)
        want, wpos = _density(fresh, seed, order, interp, positions)
        fresh.close()
        assert np.abs((got - want) / (2 + want)).max() < 2e-6, (order, interp)
        assert abs(got.mean()) < 1e-5
        if positions:
            assert np.array_equal(gpos, wpos)
    ctx.close()
