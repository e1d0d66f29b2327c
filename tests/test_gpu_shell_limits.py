"""Limits of the normalisation: what is refused for too many shells.

The redshift table is stretched so that z(L/2), and with it the number of
shells, is far beyond any survey's.
"""
import numpy as np
import pytest

from conftest import make_run
from test_gpu_shells import POPS

pytestmark = pytest.mark.gpu


def _context(workdir, nz, ntr):
    """A 32^3 context whose normalisation has nz shells."""
    from colore_amd import lib
    N = 32
    _, run = make_run("C2", N, workdir, z_max=1.2, with_maps=False, populations=tuple(POPS[ntr]))
    L = run.scalar("l_box")
    ta = run.table_arrays()
    ta["z"] = ta["z"] * (0.05 * (nz - 1.5) / np.interp(0.5 * L, ta["r"], ta["z"]))
    ctx = lib.Context(N, L)
    ctx.upload_table_arrays(ta)
    for i in range(ntr):
        amp, bz, model = run.tracer(0, i)
        ctx.set_tracer(0, i, model, amp, bz)
    return ctx


# eight tracers: four wavefronts of (nz + 64) shells of ten sums in 160 KB
@pytest.mark.parametrize("nz,ntr,ok", [(444, 8, True), (445, 8, False), (600, 8, False), (1024, 1, True), (1025, 1, False)])
def test_shells_times_tracers(workdir, nz, ntr, ok):
    ctx = _context(workdir, nz, ntr)
    s2 = ctx.gaussian_fields(3, 2.0, True)
    if ok:
        n, cnt, _, _ = ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=ntr, cap=1024)
        assert n == nz and 0 < cnt.sum() <= 32 ** 3
    else:
        with pytest.raises(RuntimeError, match="shells"):
            ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=ntr, cap=1200)
    ctx.close()


def test_ensemble_shells(workdir):
    """An ensemble's contexts have the same limit (the captured pass has no check of its own)."""
    from colore_amd import lib
    ctx = _context(workdir, 1025, 1)
    with pytest.raises(RuntimeError, match="shells"):
        lib.Ensemble([ctx], src_cap=1000)
    ctx.close()
