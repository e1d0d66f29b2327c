"""1LPT densities where the device has room for the displacement grids but not
for the tiles' regions: the same density (deposits add in an order that varies:
2e-6 of 1 + delta, as in test_lpt_calls_in_turn)."""
import numpy as np
import pytest

from conftest import make_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,interp", [(512, 1), (512, 2)])
def test_lpt_without_room_for_regions(workdir, N, interp):
    from colore_amd import lib
    from device_memory import free_bytes, only
    _, run = make_run("C2", N, workdir, z_max=0.6, with_maps=False)
    ctx = lib.Context(N, run.scalar("l_box"))
    ctx.upload_tables(run.tables())

    def density():
        ctx.gaussian_fields(3, 2.0, True)
        ctx.lpt_density(interp, 1)
        return ctx.fetch_grid(0)[:, :, :N].astype(np.float64)

    def fresh_memory():
        nonlocal ctx
        ctx.close()
        ctx = lib.Context(N, run.scalar("l_box"))
        ctx.upload_tables(run.tables())
        ctx.gaussian_fields(3, 2.0, True)
        ctx.synchronize()

    want = density()
    fresh_memory()
    grid = N * N * ((N + 2 + 31) // 32 * 32) * 4
    regions = (N // 16) ** 3 * 20 ** 3 * 4
    room = 3 * grid + regions // 2
    with only(room):
        free = free_bytes()
        assert 3 * grid < free < 3 * grid + regions, (free, grid, regions)
        got = density()
    ctx.close()
    assert np.abs((got - want) / (2 + want)).max() < 2e-6
    assert abs(got.mean()) < 1e-5
