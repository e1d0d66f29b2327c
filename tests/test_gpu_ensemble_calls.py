"""Single calls on the contexts of a captured ensemble, between its replays.

A captured graph holds its contexts' buffers by address, and the single calls
that a flagged realisation is re-run with share (and may grow) those buffers.
After any of them the ensemble's next run must again equal single runs on fresh
contexts bit for bit: sampling at the same sizes leaves every buffer where it
is, a larger catalogue, map, list or base-pixel table has the graph captured
again.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NSIDE = 32


def _ensemble(workdir, src_cap):
    from colore_amd import inputs, lib
    from test_gpu_ensemble import _contexts
    # two of the workload's smallest boxes, with a population that lies inside them
    rs = [dict(r, nz_mean=0.06) for r in inputs.c4_realisations(64, 4000) if r["n_grid"] == 128][:2]
    runs, ctxs = _contexts(rs, workdir)
    rk = np.array([run.scalar("r_max") for run in runs])
    ens = lib.Ensemble(ctxs, src_cap=src_cap, nside_kappa=NSIDE, r_kappa=rk, nstreams=2)
    seeds = np.array([r["seed"] for r in rs], dtype=np.uint32)
    rsm = np.array([run.scalar("r_smooth") for run in runs])
    return rs, runs, ctxs, ens, seeds, rsm


def _single_calls(ctx, run, seed, nside_base=2):
    s2 = ctx.gaussian_fields(seed, run.scalar("r_smooth"), True)
    ctx.shell_norms(lognormal_fused=True, sigma2=s2, ntracers=1)
    return ctx.sample_sources(-1, seed, nside_base)


def test_single_calls_between_replays(workdir):
    from test_gpu_ensemble import _check, _single
    rs, runs, ctxs, ens, seeds, rsm = _ensemble(workdir, 4_000_000)
    wants = [_single(run, r, NSIDE) for run, r in zip(runs, rs)]
    assert all(len(w[1]) > 1000 for w in wants)

    def run_and_check():
        bad, _ = ens.run(seeds, rsm)
        assert bad == 0
        for i in range(len(rs)):
            _check(ens, ctxs, i, wants[i])

    run_and_check()
    # the same sizes: nothing moves
    held = ctxs[0].lib.clr_device_bytes(ctxs[0].h)
    assert _single_calls(ctxs[0], runs[0], 5) > 0
    assert ctxs[0].lib.clr_device_bytes(ctxs[0].h) == held
    run_and_check()
    # a map that outgrows the scratch the graph's lists lie in
    held = ctxs[1].lib.clr_device_bytes(ctxs[1].h)
    _single_calls(ctxs[1], runs[1], 6)
    ctxs[1].kappa(256, np.array([runs[1].scalar("r_max")]))
    assert ctxs[1].lib.clr_device_bytes(ctxs[1].h) > held
    run_and_check()
    # another base-pixel table
    _single_calls(ctxs[0], runs[0], 7, nside_base=8)
    run_and_check()
    run_and_check()
    ens.close()
    for c in ctxs:
        c.close()


def test_flagged_realisation_rerun(workdir):
    """A catalogue past src_cap is flagged, re-run with the single calls (which
    grow it), and fits in the next run of the ensemble."""
    from test_gpu_ensemble import _check, _single
    rs, runs, ctxs, ens, seeds, rsm = _ensemble(workdir, 1000)
    wants = [_single(run, r, NSIDE) for run, r in zip(runs, rs)]
    bad, _ = ens.run(seeds, rsm)
    assert bad == 2 and all(ens.result(i)[1] & 4 for i in range(2))
    for i in range(2):
        assert _single_calls(ctxs[i], runs[i], rs[i]["seed"]) == len(wants[i][1])
        pos, ipix = ctxs[i].fetch_sources(0, len(wants[i][1]))
        assert np.array_equal(pos, wants[i][1]) and np.array_equal(ipix, wants[i][2])
    for _ in range(2):
        bad, _ = ens.run(seeds, rsm)
        assert bad == 0
        for i in range(2):
            _check(ens, ctxs, i, wants[i])
    ens.close()
    for c in ctxs:
        c.close()


def test_fields_call_before_a_replay(workdir):
    """clr_gaussian_fields returns while the potential's last passes run on the
    context's second stream; a replay that follows at once must wait for them."""
    from test_gpu_ensemble import _check, _single
    rs, runs, ctxs, ens, seeds, rsm = _ensemble(workdir, 4_000_000)
    wants = [_single(run, r, NSIDE) for run, r in zip(runs, rs)]
    for rep in range(3):
        bad, _ = ens.run(seeds, rsm)
        assert bad == 0
        for i in range(len(rs)):
            _check(ens, ctxs, i, wants[i])
        for c, run in zip(ctxs, runs):
            c.gaussian_fields(100 + rep, run.scalar("r_smooth"), True)
    ens.close()
    for c in ctxs:
        c.close()
