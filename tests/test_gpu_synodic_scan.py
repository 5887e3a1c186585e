"""GPU: the multi-pass section detection's division-free scan against the
one-wave kernel, which walks every segment."""

import numpy as np
import pytest
import torch

from hiten_amd import synodic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 3, 62, 63, 64, 65, 245, 246, 489, 490, 491, 1000])
def test_scan_misses_no_segment(gpu, m):
    """Lengths around the scan's chunks and parts: noisy values close to the
    plane, touches without a sign change at the samples (two roots inside a
    segment), samples on the plane, NaN and infinite samples, times that repeat
    or go back, in every option set."""
    rng = np.random.default_rng(m)
    n = 40
    k = np.arange(m)
    X = rng.normal(size=(n, m, 6))
    for i in range(n):
        level = 10.0 ** rng.uniform(-3, 0)
        y = level * (1.5 + np.sin(0.05 * k + i))           # above the plane
        at = rng.random(m) < 0.02
        kind = i % 5
        if kind == 0:
            y[at] *= -1.0
        elif kind == 1:
            y[at] = 0.0
        elif kind == 2:                                     # dips between samples
            y[at] = 1e-3 * level * rng.random(at.sum())
        elif kind == 3:
            y[at] *= 1e-14 * rng.choice([-1.0, 1.0], at.sum())
        else:
            y = level * rng.normal(size=m) + 4.0 * level
        X[i, :, 1] = y
    X[5, rng.integers(m), 1] = np.nan
    X[6, rng.integers(m), 1] = np.inf
    X[7, rng.integers(m), 3] = np.nan
    T = np.cumsum(rng.uniform(0.5, 1.5, (n, m)), axis=1)
    for i in (2, 7, 12, 20):                                # times that repeat or go back
        j = rng.integers(m, size=max(1, m // 40))
        T[i, j] = T[i, np.maximum(j - 1, 0)] - (i % 3)
    lengths = rng.integers(max(0, m - 3), m + 1, n).astype(np.int32)
    for opt in (dict(interp_kind="cubic", segment_refine=7), dict(interp_kind="cubic"),
                dict(interp_kind="linear", segment_refine=3),
                dict(interp_kind="cubic", segment_refine=7, direction=-1),
                dict(interp_kind="cubic", segment_refine=2, tol_on_surface=1e-2, direction=1),
                dict(interp_kind="linear", offset=0.01)):
        a, b = (synodic.detect_arrays(T, X, normal=synodic.axis_normal("y"), lengths=lengths,
                                      newton_max_iter=5, two_pass=two, **opt)
                for two in (False, True))
        assert torch.equal(a.count, b.count)
        cap = min(a.t.shape[1], b.t.shape[1])
        held = torch.arange(cap, device=a.t.device) < a.count[:, None]
        assert torch.equal(a.t[:, :cap][held].nan_to_num(7.0), b.t[:, :cap][held].nan_to_num(7.0))
        assert torch.equal(a.x[:, :cap][held].nan_to_num(7.0), b.x[:, :cap][held].nan_to_num(7.0))
