"""GPU: end states with the layout left open, recorded into a HIP graph."""

import numpy as np
import pytest
import torch

from hiten_amd import batch, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [100, 4097])
def test_captured_auto_layout_replays(gpu, n):
    """42-d, on either side of the layout's size rule: every replay, on replaced
    inputs and with eager work between, against the eager call."""
    rng = np.random.default_rng(n)

    def inputs():
        x = W.with_identity_stm(W.planar_seeds(rng, n))
        return (torch.as_tensor(x, device=gpu),
                torch.as_tensor(rng.uniform(0.05, 0.5, n), device=gpu))

    y, tf = inputs()
    mu = torch.full((n,), W.MU_EM, dtype=torch.float64, device=gpu)
    t0 = torch.zeros(n, dtype=torch.float64, device=gpu)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        batch.dop853_final(mu, y, t0, tf, dim=42)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        r = batch.dop853_final(mu, y, t0, tf, dim=42)
    for _ in range(4):
        y2, tf2 = inputs()
        y.copy_(y2)
        tf.copy_(tf2)
        g.replay()
        torch.cuda.synchronize()
        want = batch.dop853_final(mu, y2, t0, tf2, dim=42)
        assert torch.equal(r.y, want.y)
        assert torch.equal(r.status, want.status)
        assert torch.equal(r.n_accepted, want.n_accepted)
