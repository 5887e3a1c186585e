"""GPU: calls launched on another stream than the current one, while the
current one still has to form their inputs, against the same calls on the
current stream."""

import numpy as np
import pytest
import torch

from hiten_amd import batch, corrector, energy, singlehit, synodic, workloads as W

pytestmark = pytest.mark.gpu
MU = W.MU_EM
DELAY = 50_000_000          # cycles of a spinning kernel: some tens of milliseconds


def _stm(y):
    eye = torch.eye(6, dtype=y.dtype, device=y.device).reshape(1, 36)
    return torch.cat([eye.expand(len(y), 36), y], dim=1)


def _tensors(r):
    if isinstance(r, torch.Tensor):
        return [r]
    return list(r) if isinstance(r, tuple) else list(vars(r).values())


CALLS = {
    "final6": (1000, lambda y, tf, s: batch.dop853_final(MU, y, 0.0, tf, stream=s)),
    "final6 one": (1, lambda y, tf, s: batch.dop853_final(MU, y, 0.0, tf, stream=s)),
    "final42 pair": (100, lambda y, tf, s: batch.dop853_final(
        MU, _stm(y), 0.0, tf, dim=42, stream=s)),
    "final42 persistent": (4097, lambda y, tf, s: batch.dop853_final(
        MU, _stm(y), 0.0, tf, dim=42, stream=s)),
    "grid6": (300, lambda y, tf, s: batch.dop853_grid(MU, y, 0.0, tf, 50, stream=s)),
    "grid6 times": (300, lambda y, tf, s: batch.dop853_grid(
        MU, y, None, None, 0, t_eval=np.linspace(0.0, 0.3, 50), stream=s)),
    "grid42": (50, lambda y, tf, s: batch.dop853_grid(
        MU, _stm(y), 0.0, tf, 20, dim=42, stream=s)),
    "event": (1000, lambda y, tf, s: batch.dop853_event(MU, y, 0.0, tf, stream=s)),
    "rk8 event": (200, lambda y, tf, s: batch.rk_fixed_event(MU, y, 0.0, tf, 100, stream=s)),
    "rk8": (200, lambda y, tf, s: batch.rk_fixed(MU, y, 0.0, tf, 100, return_derivatives=True,
                                                 stream=s)),
    "field": (1000, lambda y, tf, s: batch.eval_rhs(MU, y, stream=s)),
    "filters": (64, lambda y, tf, s: energy.traj_filters(y.repeat(30, 1, 1).transpose(0, 1), MU,
                                                         stream=s)),
}


@pytest.mark.parametrize("name", list(CALLS))
def test_other_stream_waits_for_its_inputs(gpu, name):
    n, call = CALLS[name]
    rng = np.random.default_rng(n)
    y = torch.as_tensor(W.planar_seeds(rng, n), device=gpu)
    tf = torch.as_tensor(rng.uniform(0.05, 0.5, n), device=gpu)
    want = [t.cpu() for t in _tensors(call(y, tf, None))]
    side = torch.cuda.Stream()
    for _ in range(2):                      # the second call takes freed memory again
        torch.cuda.synchronize()
        torch.cuda._sleep(DELAY)
        got = _tensors(call(y * 1.0, tf * 1.0, side))
        # what the call has let go of may be handed out again only after it
        junk = [torch.full((k,), -1, dtype=torch.int32, device=gpu)
                for k in (1, n, 2 * n, 12 * n, 84 * n)]
        side.synchronize()
        for g, w in zip(got, want):
            assert torch.equal(g.cpu(), w)
        del junk


def _corrections(y, s):
    ps = [corrector.halo_problem(MU, [0.8234, 0, 0.0224 + 1e-5 * i, 0, 0.1343, 0],
                                 max_attempts=10) for i in range(5)]
    return np.array([[*r.x_corrected, r.half_period, r.n_stm]
                     for r in corrector.correct_device(ps, stream=s)])


def _sections(y, s):
    a = torch.linspace(0.0, 40.0, 900, dtype=y.dtype, device=y.device)
    X = torch.sin(a)[None, :, None] + y[:, None, :]
    r = synodic.detect_arrays(a, X, normal=synodic.axis_normal("y"), cap=2, stream=s)
    torch.cuda.synchronize()                # the hits beyond the counts are not written
    return np.array([[h.time for h in row] for row in synodic.hits_from_arrays(r)])


def _crossings(y, s):
    plane = singlehit._PlaneEvent("y", 0.0, None)
    ok, t, x = singlehit.plane_crossing_device(MU, y.cpu().numpy(), plane, 1, (0.0, 3.1),
                                               (1.4, 3.1), stream=s)
    return np.column_stack([ok, t, x])


@pytest.mark.parametrize("call", [_corrections, _sections, _crossings])
def test_results_read_on_the_host_are_the_other_streams(gpu, call):
    y = torch.as_tensor(W.planar_seeds(np.random.default_rng(2), 40), device=gpu)
    want = call(y, None)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(DELAY)            # the kernel starts late
    np.testing.assert_array_equal(call(y, side), want)


def test_capture_on_another_stream_than_the_current(gpu):
    """The launch stream records and the current one does not: the kernel is
    recorded as it stands, and every replay runs it."""
    n = 4097
    rng = np.random.default_rng(3)
    y = _stm(torch.as_tensor(W.planar_seeds(rng, n), device=gpu))
    tf = torch.as_tensor(rng.uniform(0.05, 0.3, n), device=gpu)
    mu = torch.full((n,), MU, dtype=torch.float64, device=gpu)
    t0 = torch.zeros(n, dtype=torch.float64, device=gpu)
    want = batch.dop853_final(mu, y, t0, tf, dim=42, variant="plain")
    side = torch.cuda.Stream()
    b = batch.prepare_final(mu, y, t0, tf, 42)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        g.capture_begin()
    batch.launch_final(b, variant="plain", stream=side)
    with torch.cuda.stream(side):
        g.capture_end()
    for _ in range(3):
        b.y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(b.result().y, want.y)
