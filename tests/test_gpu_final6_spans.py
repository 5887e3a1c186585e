"""GPU: 6-d end states dealt out by span within a workgroup against the same
batch in plain order and against the oracle."""

import numpy as np
import pytest
import torch

from hiten_amd import batch, workloads as W

pytestmark = pytest.mark.gpu
MU = W.MU_EM


@pytest.mark.parametrize("n", [98305, 114687, 114688, 131071, 131073])
def test_dealing_by_span_changes_no_result(gpu, oracle, n):
    """Both workgroup sizes, whole and partly filled: spans that differ, repeat
    and are zero, reversed or too small to sort, an attempt limit, backward."""
    rng = np.random.default_rng(n)
    y = W.planar_seeds(rng, n)
    y[:, 1:3] = rng.uniform(-0.02, 0.02, (n, 2))
    tf = rng.uniform(0.01, 0.3, n)
    tf[rng.integers(n, size=500)] = 0.0
    tf[rng.integers(n, size=500)] = -0.2
    tf[rng.integers(n, size=500)] = 0.25
    tf[rng.integers(n, size=500)] = 0.25 * (1.0 + 1e-9)
    tf[rng.integers(n, size=50)] = 1e-12
    tf[-1] = 0.3
    for fwd, steps in ((1, 1_000_000), (-1, 1_000_000), (1, 3)):
        kw = dict(forward=fwd, variant="plain", max_steps=steps)
        a = batch.dop853_final(MU, y, 0.0, tf, **kw)
        b = batch.dop853_final(MU, y, 0.0, tf, block=128, **kw)
        for u, v in zip(vars(a).values(), vars(b).values()):
            assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())
    sys = oracle.System("cr3bp6", mu=MU)
    r = batch.dop853_final(MU, y, 0.0, tf, variant="plain")
    yr = r.y.cpu().numpy()
    for i in (0, n // 2, n - 1):
        if tf[i] > 0.0:
            want = oracle.dop853(sys, y[i], np.array([0.0, tf[i]]), rtol=1e-12, atol=1e-12,
                                 max_step=1e4)[0][-1]
            assert np.array_equal(yr[i], want)


@pytest.mark.parametrize("per_cu,more", [(384, 0), (384, 1), (448, -1), (448, 0), (512, 0),
                                         (512, 1)])
def test_lines_of_the_rule_on_this_device(gpu, per_cu, more):
    """Either side of every line of the rule, which lie by the device's CUs."""
    n = per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more
    rng = np.random.default_rng(n)
    y = W.planar_seeds(rng, n)
    tf = rng.uniform(0.01, 0.2, n)
    a = batch.dop853_final(MU, y, 0.0, tf, variant="plain")
    b = batch.dop853_final(MU, y, 0.0, tf, variant="plain", block=128)
    for u, v in zip(vars(a).values(), vars(b).values()):
        assert torch.equal(u, v)
