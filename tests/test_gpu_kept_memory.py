"""Memory that a context keeps between calls does not cost other calls theirs.

A 2LPT call leaves its eight grids with the context.  With the rest of the
device filled, a convergence map must still take its per-cell records where they
fit a quarter of the memory that is free or kept, and a catalogue that needs the
kept memory must be sampled, with the results of an unfilled device.
"""
import numpy as np
import pytest

from conftest import make_run
from device_memory import free_bytes, only

pytestmark = pytest.mark.gpu

N = 512


def _lpt_context(workdir, **kw):
    from colore_amd import lib
    _, run = make_run("C2", N, workdir, z_max=0.6, with_maps=False, **kw)
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())
    amp, bz, model = run.tracer(0, 0)
    ctx.set_tracer(0, 0, model, amp, bz)
    before = ctx.lib.clr_device_bytes(ctx.h)
    ctx.gaussian_fields(3, 2.0, True)
    ctx.lpt_density(1, 2)
    kept = 8 * N * N * ((N + 2 + 31) // 32 * 32) * 4
    assert ctx.lib.clr_device_bytes(ctx.h) > before + kept
    return run, ctx, kept, (amp, bz, model)


def test_records_beside_kept_grids(workdir):
    run, ctx, kept, _ = _lpt_context(workdir)
    r = np.array([run.scalar("r_max")])
    records = 24 * N ** 3
    with only(4 * records - kept // 2):
        free = free_bytes()
        assert free < 4 * records < free + kept, (free, kept, records)
        before = ctx.lib.clr_device_bytes(ctx.h)
        got = ctx.kappa(512, r)
        assert ctx.lib.clr_device_bytes(ctx.h) >= before + records
    assert np.array_equal(got, ctx.kappa(512, r))
    ctx.close()


def test_catalogue_takes_kept_memory(workdir):
    run, ctx, kept, (amp, bz, model) = _lpt_context(workdir)
    ctx.shell_norms(lognormal_fused=False, ntracers=1)
    tab = ctx.norm_table(0, 0)

    def sample(scale):
        ctx.set_tracer(0, 0, model, amp * scale, bz)
        ctx.set_norm_table(0, 0, *tab)
        return ctx.sample_sources(0, 11, 2)

    n = sample(1e-2)
    scale = 1e-2 * 3e7 / n   # about 3e7 sources, 600 MB
    with only(200 << 20):
        assert free_bytes() < 500 << 20
        n = sample(scale)
        assert n * 20 > 500 << 20 and n * 20 < kept
        pos, ipix = ctx.fetch_sources(0, n)
    assert sample(scale) == n
    pos2, ipix2 = ctx.fetch_sources(0, n)
    assert np.array_equal(pos, pos2) and np.array_equal(ipix, ipix2)
    ctx.close()
