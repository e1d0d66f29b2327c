"""The shell pass's tilings against the FP64 oracle.

compute_density_normalization (density.c:1128-1393) runs on tiles chosen from
the cell size, the shells' width and the number of tracers: single rows of
4 x 4 x 4 cells (deep boxes of few cells, with several passes per tile where a
tile spans more than four shells), 8 x 4 x 8 cells, and 16 x 8 x 4 or
16 x 16 x 4 cells with the tables staged in LDS.  Every one of them must give
the oracle's cell counts exactly and its z and bias sums to the rounding of
FP32 terms (2e-6, as in test_shell_norms), with the lognormal transform fused
or not, and the same bits on every call.
"""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu

G = ("gauss", 0.3, 0.1, 1e-4)
POPS = {1: [(G, ("const", 1.3), "exponential")],
        2: [(G, ("1+z",), "exponential"), (G, ("const", 1.5), "exp-truncated")],
        3: [(G, ("1+z",), "exponential"), (G, ("const", 1.5), "exp-truncated"), (G, ("const", 2.2), "truncated")],
        8: [(G, ("const", 0.5 + 0.3 * i), ("exponential", "exp-truncated", "truncated")[i % 3]) for i in range(8)]}


@pytest.mark.parametrize("N,z_max,ntr", [
    (32, 6.0, 2),     # cells of several shells: passes of four shells
    (64, 1.6, 8),     # 4 x 4 x 4, the widest window of sums
    (192, 1.2, 3),
    (128, 0.4, 1),    # 8 x 4 x 8
    (192, 0.5, 3),
    (384, 1.2, 2),    # 16 x 8 x 4
    (384, 1.2, 1),    # 16 x 16 x 4
])
def test_shell_tiles(workdir, N, z_max, ntr):
    from colore_amd import lib
    from oracle_lib import Oracle
    _, run = make_run("C2", N, workdir, z_max=z_max, with_maps=False, populations=tuple(POPS[ntr]))
    L = run.scalar("l_box")
    ctx = lib.Context(N, L)
    ctx.upload_tables(run.tables())
    tracers = [run.tracer(0, i) for i in range(ntr)]
    for i, (amp, bz, model) in enumerate(tracers):
        ctx.set_tracer(0, i, model, amp, bz)
    s2 = ctx.gaussian_fields(77, 3.0, True)
    g0 = ctx.fetch_grid(0).astype(np.float64)
    nz, cnt, zs, sums = ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=ntr)
    gl = ctx.fetch_grid(0)
    orc = Oracle(run.table_arrays())
    ol = orc.density(N, L, g0, s2, 0)
    assert np.abs(gl[:, :, :N] - ol[:, :, :N]).max() / (1 + np.abs(ol).max()) < 1e-6
    onz, _, ocnt, ozs, osums = orc.shell_sums(N, L, gl.astype(np.float64), [(b, m) for _, b, m in tracers])
    assert nz == onz and np.array_equal(cnt, ocnt)
    np.testing.assert_allclose(zs, ozs, rtol=2e-6)
    np.testing.assert_allclose(sums, osums, rtol=2e-6)
    for noalloc in (False, True):
        if noalloc and nz * (2 + ntr) > 320:
            continue
        _, c2, z2, u2 = ctx.shell_norms(lognormal_fused=False, sigma2=s2, ntracers=ntr, noalloc=noalloc)
        assert np.array_equal(c2, cnt) and np.array_equal(z2, zs) and np.array_equal(u2, sums)
    ctx.close()
