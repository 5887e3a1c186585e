"""The bounds of the waits in the persistent pair form's scheduler
(hh_dop853_final_bounded): with waits of no or few polls every wave still ends,
and a trajectory either has the plain kernel's results or says it was dropped."""

import numpy as np
import pytest

from hiten_amd import _lib, batch, workloads as W


def _bounded(b, polls, max_steps=200_000):
    lib = _lib.load()
    ws, size = b.workspace_for(_lib.HH_VARIANT_PERSISTENT_PAIR)
    rc = lib.hh_dop853_final_bounded(
        polls, b.n, 42, batch._ptr(b.mu), batch._ptr(b.t0), batch._ptr(b.tf), 1e-12, 1e-12, 1e4,
        batch.MIN_STEP, max_steps, 1, 0, batch._ptr(b.y0), batch._ptr(b.y), batch._ptr(b.status),
        batch._ptr(b.n_accepted), batch._ptr(b.n_rejected), _lib.HH_VARIANT_PERSISTENT_PAIR, 0, 0,
        ws, size, batch._ptr(b.order), _lib.stream_handle())
    _lib.check(rc, "hh_dop853_final_bounded")
    return [t.cpu().numpy() for t in vars(b.result()).values()]


def test_negative_bound_is_refused():
    lib = _lib.load(require_gpu=False)
    rc = lib.hh_dop853_final_bounded(-1, 4, 42, None, None, None, 1e-12, 1e-12, 1e4, 1e-15, 10, 1,
                                     0, None, None, None, None, None, 4, 0, 0, None, 0, None, None)
    assert rc == _lib.HH_ERR_ARGS and b"wait_polls" in lib.hh_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("polls", [1 << 22, 3, 0])
@pytest.mark.parametrize("heavy,pair,exclusive", [(3, 0, 0), (3, 3, 0), (3, 3, 1), (3, 60, 3)])
def test_every_wave_ends_and_no_loss_is_silent(gpu, polls, heavy, pair, exclusive):
    print(f"\n[case] {polls} polls, heavy={heavy} pair={pair} exclusive={exclusive}", flush=True)
    w = W.stm_uneven(n=2048)
    plain = batch.dop853_final(w["mu"], w["y0"], w["t0"], w["tf"], dim=42, variant="plain",
                               max_steps=200_000)
    want = [t.cpu().numpy() for t in vars(plain).values()]
    saved = _lib.set_tuning(heavy_projected=heavy, min_age=1, pair_projected=pair,
                            exclusive_projected=exclusive)
    try:
        y, status, nacc, nrej = _bounded(
            batch.prepare_final(w["mu"], w["y0"], w["t0"], w["tf"], 42), polls)
    finally:
        _lib.set_tuning(**saved)
    lost = status == 4                       # HH_STATUS_DROPPED
    assert not (polls == 1 << 22 and lost.any())
    assert (nacc[lost] == 0).all() and (nrej[lost] == 0).all()
    for g, e in zip((y, status, nacc, nrej), want):
        assert np.array_equal(g[~lost], e[~lost])
    print(f"[case] dropped {lost.sum()}", flush=True)
