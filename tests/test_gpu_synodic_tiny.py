"""GPU: plane values so small that the product of two of one sign rounds to 0,
which the reference counts as a crossing: the multi-pass
detection against the one-wave kernel and the oracle."""

import numpy as np
import pytest
import torch

from hiten_amd import synodic
from oracle import synodic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level", [1e-140, 3e-151, 1e-154, 1e-161, 1e-162, 1e-163, 1e-200, 1e-300])
@pytest.mark.parametrize("refine", [0, 3])
def test_products_that_vanish_are_crossings(gpu, level, refine):
    """Smooth positive values, whose interpolant stays far from the plane in
    their own scale, on lengths around the scan's chunks."""
    m = 130
    t = np.linspace(0.0, 13.0, m)
    X = np.ones((3, m, 6))
    X[:, :, 0] = np.arange(m)                # section points that differ
    for i in range(3):
        X[i, :, 1] = level * (2.0 + 0.1 * np.sin(0.3 * np.arange(m) + i))
    X[1, :, 1] *= -1.0
    X[2, 70:, 1] *= 1e160                    # leaves the range half way
    for kind in ("linear", "cubic"):
        kw = dict(interp_kind=kind, segment_refine=refine, tol_on_surface=0.0)
        a, b = (synodic.hits_from_arrays(synodic.detect_arrays(
                    t, X, normal=synodic.axis_normal("y"), two_pass=two, cap=m,
                    plane_coords=("x", "vx"), **kw))
                for two in (False, True))
        for i in range(3):
            assert [h.time for h in a[i]] == [h.time for h in b[i]]
            assert all(np.array_equal(u.state, v.state) for u, v in zip(a[i], b[i]))
        if refine == 0:
            for i in range(3):
                want = S.detect(t, X[i], normal=synodic.axis_normal("y"), plane_idx=(0, 3),
                                **kw)
                assert [h.time for h in b[i]] == [w[0] for w in want]
            assert bool(b[0]) == (level < 1e-162)
