"""Custom maps of densities that are not all finite.

A cell's infinite density reaches a step through its trilinear weight, and bias
models turn it into an infinite, zero or finite value (b > 0, b < 0, b = 0): the
map has the oracle's infinities and NaN in the oracle's pixels, and its values
elsewhere (1e-5 of their RMS, as in test_custom_map).
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nside", [4, 256])   # several lanes per pixel, one
@pytest.mark.parametrize("model,b", [(0, 1.5), (0, -0.7), (0, 0.0), (1, 1.5), (2, 2.2)])
def test_infinite_densities(workdir, nside, model, b):
    from colore_amd import lib
    from oracle_lib import Oracle
    N = 64
    _, run = make_run("C2", N, workdir, z_max=1.0, with_maps=False)
    L = run.scalar("l_box")
    ctx = lib.Context(N, L)
    ctx.upload_tables(run.tables())
    rng = np.random.default_rng(8)
    dens = np.zeros(ctx.padded_shape, dtype=np.float32)
    cells = np.expm1(rng.normal(0, 0.5, (N, N, N))).astype(np.float32)
    pick = rng.random((N, N, N))
    cells[pick < 2e-4] = np.inf
    cells[(pick > 0.5) & (pick < 0.5001)] = np.nan
    cells[pick > 0.98] = -1
    dens[:, :, :N] = cells
    ctx.upload_grid(lib.CLR_GRID_DENS, dens)
    ctx.declare_grids(0.2, True)
    r = run.table_arrays()["r"]
    kz, bz, norm = np.ones_like(r), np.full_like(r, b), np.ones_like(r)
    ctx.set_tracer(lib.CLR_TRACER_CSTM, 0, model, kz, bz)
    ctx.set_norm_table(lib.CLR_TRACER_CSTM, 0, norm, 1.0, 1.0)
    out = ctx.custom_map(0, nside).astype(np.float64)
    ctx.close()
    want = Oracle(run.table_arrays()).cstm(N, L, dens.astype(np.float64), kz, bz, norm, 1.0, 1.0, model, nside)
    assert np.array_equal(np.isnan(out), np.isnan(want))
    assert np.array_equal(np.isposinf(out), np.isposinf(want)) and np.array_equal(np.isneginf(out), np.isneginf(want))
    ok = np.isfinite(want)
    assert 0.1 < ok.mean()
    rms = np.sqrt(np.mean(want[ok] ** 2))
    assert np.abs(out[ok] - want[ok]).max() <= 1e-5 * rms
