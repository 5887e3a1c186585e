"""GPU: every kept arc of a manifold has memory of its own, so that one arc
kept does not hold the others."""

import numpy as np
import pytest
import torch

from hiten_amd import manifold as M, workloads as W

pytestmark = pytest.mark.gpu


def _root(a):
    while isinstance(a.base, np.ndarray):
        a = a.base
    return a


@pytest.mark.parametrize("method", ["adaptive", "fixed"])
def test_kept_arcs_share_no_memory(gpu, method):
    state = [0.8234, 0.0, 0.0224, 0.0, 0.1343, 0.0]
    r = M.compute_manifold(W.MU_EM, state, 2.74, method=method, step=0.1, dt=1e-2,
                           energy_tol=np.inf, safe_distance=0.0, stm_steps=200)
    assert r.successes > 1 and r.successes == len(r.states_list) == len(r.times_list)
    for i, a in enumerate(r.states_list):
        assert a.shape == (len(r.times_list[i]), 6) and a.flags.c_contiguous and a.flags.writeable
        assert _root(a).nbytes == a.nbytes and a.flags.owndata
        assert not any(np.shares_memory(a, b) for b in r.states_list[:i])
    before = r.states_list[1].copy()
    r.states_list[0][:] = 0.0
    assert np.array_equal(r.states_list[1], before)


@pytest.mark.parametrize("n,m", [(1, 2), (5, 300), (3, 50_000), (40, 4713), (23, 4369)])
def test_rows_in_chunks(gpu, n, m):
    """One row a chunk (2.4 MB), chunks that divide the rows and that do not, some
    and all of the rows, from a permuted view too."""
    x = torch.randn((m, 6, n), dtype=torch.float64, device=gpu)
    for states in (x.permute(2, 0, 1), x.permute(2, 0, 1).contiguous()):
        host = states.cpu().numpy()
        for idx in (np.arange(n), np.arange(n)[::2], np.arange(n)[:0]):
            got = M._host_rows(states, idx)
            assert len(got) == len(idx)
            assert all(np.array_equal(g, host[i]) for g, i in zip(got, idx))
