"""GPU: the device-resident corrector's rounds -- those whose speculative STM is
taken, dropped because the state has converged or is turned down by the line
search, or integrated afterwards -- alone and with more corrections than the
chip holds at once, against the host-driven bank and against each other."""

import numpy as np
import pytest

from hiten_amd import corrector as Cr, workloads as W

pytestmark = pytest.mark.gpu
MU = W.MU_EM
TOL_X = 1e-10


@pytest.mark.parametrize("copies", [1, 100])
def test_rounds_with_and_without_their_stm(gpu, copies):
    seed = [0.8234, 0, 0.0224, 0, 0.1343, 0]
    done = Cr.correct_device([Cr.halo_problem(MU, seed, max_attempts=20)])[0]
    assert done.converged
    ps = [Cr.halo_problem(MU, seed, max_attempts=20),
          Cr.halo_problem(MU, list(done.x_corrected), max_attempts=20),     # ends at once
          Cr.halo_problem(MU, seed, max_attempts=1),                        # before the last STM
          Cr.halo_problem(MU, [0.84, 0, 0.1, 0, 0.22, 0], max_attempts=20),
          Cr.halo_problem(MU, [0.86, 0, 0.17, 0, 0.28, 0], max_attempts=6),
          Cr.halo_problem(MU, seed, max_attempts=20, armijo_c=0.95),        # trials turned down
          Cr.lyapunov_problem(MU, [0.83, 0, 0, 0, 0.08, 0], max_attempts=12),
          Cr.halo_problem(MU, [3.0, 0, 0.0, 0, 0.0, 0.0], max_attempts=5)]  # no crossing
    got = Cr.correct_device(ps * copies)
    want = Cr.correct_batch(ps)
    for i, w in enumerate(want):
        g = got[i]
        assert g.converged == w.converged
        assert g.error.split(" ")[0] == w.error.split(" ")[0]
        if w.converged:
            assert np.max(np.abs(g.x_corrected - w.x_corrected)) <= TOL_X
            assert abs(g.half_period - w.half_period) <= TOL_X
        for c in range(1, copies):
            h = got[c * len(ps) + i]
            assert np.array_equal(h.x_corrected, g.x_corrected, equal_nan=True)
            assert (h.iterations, h.n_event_searches, h.n_stm) == \
                (g.iterations, g.n_event_searches, g.n_stm)
    assert got[1].iterations == 0 and got[1].n_stm == 0
