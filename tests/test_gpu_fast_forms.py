"""GPU: the field and the step loops at the edges of the exponent range in
which divisions and powers take their unscaled forms (squared distances in
[2^-100, 2^100), coordinates and masses 0 or at least 2^-301, error scales in
[2^-300, 2^960)), against the oracle bit for bit: states inside, on either
side of each bound, and both in one wave."""

import numpy as np
import pytest

from hiten_amd import batch, workloads as W

pytestmark = pytest.mark.gpu

MU = W.MU_EM
#: magnitudes on both sides of the bounds 2^-301, 2^-50 (distance), 2^50
SIZES = [0.0, -0.0, 5e-324, 1e-300, 2.0 ** -302, 2.0 ** -301, 2.0 ** -300, 1e-60, 2.0 ** -51,
         2.0 ** -50, 2.0 ** -49, 1e-9, 1e-3, 2.0 ** 49, 2.0 ** 50, 2.0 ** 51]


def _states():
    rng = np.random.default_rng(5)
    rows = []
    for mu in (MU, 0.0, 2.0 ** -302, 2.0 ** -300, 3.0035e-6):
        for k, s in enumerate(SIZES):
            t = SIZES[(k + 5) % len(SIZES)]
            near = rng.uniform(0.8, 0.9)
            v = rng.normal(size=3)
            rows += [(mu, [near, 0.01, s, *v]), (mu, [near, s, t, *v]),
                     (mu, [-mu + s, 0.0, 0.0, *v]), (mu, [1.0 - mu + s, 0.0, t, *v]),
                     (mu, [1.0 - mu, s, 0.0, *v]), (mu, [s, s, s, *v])]
    mus = np.array([r[0] for r in rows])
    y = np.array([r[1] for r in rows])
    # a collision (distance 0) has no finite derivative
    d = np.minimum(np.hypot(np.hypot(y[:, 0] + mus, y[:, 1]), y[:, 2]),
                   np.hypot(np.hypot(y[:, 0] - (1.0 - mus), y[:, 1]), y[:, 2]))
    return mus[d > 0], y[d > 0]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("dim", [6, 42])
def test_field_at_the_range_bounds(gpu, oracle, dim, mixed):
    mu, x = _states()
    rng = np.random.default_rng(6)
    if mixed:
        # one edge state among states near L1 in every wave
        keep = np.arange(len(x)) % (8 if dim == 42 else 64) == 3
        x[~keep] = W.planar_seeds(rng, int((~keep).sum()))
        mu[~keep] = MU
    y = x if dim == 6 else np.concatenate([rng.normal(size=(len(x), 36)), x], axis=1)
    got = batch.eval_rhs(mu, y, dim=dim).cpu().numpy()
    f = oracle.crtbp_accel if dim == 6 else oracle.var_equations
    want = np.array([f(s, m) for s, m in zip(y, mu)])
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("dim,variant", [(6, "plain"), (6, "wide"), (42, "plain"), (42, "wide"),
                                         (42, "pair"), (42, "persistent")])
@pytest.mark.parametrize("n", [1, 9, 130])
def test_integration_at_the_range_bounds(gpu, oracle, dim, variant, n):
    """Arcs with out-of-plane motion from 0 to below the bounds, masses on both
    sides of theirs, one error scale below its bound."""
    rng = np.random.default_rng(n)
    x = W.planar_seeds(rng, n)
    tiny = np.array([0.0, 1e-300, 2.0 ** -302, 2.0 ** -300, 1e-30, 1.0])
    x[:, 2] *= tiny[np.arange(n) % 6]
    x[:, 5] = tiny[(np.arange(n) + 2) % 6] * 1e-2
    mu = np.array([MU, 0.0, 2.0 ** -302, 1e-80])[np.arange(n) % 4]
    y0 = x if dim == 6 else W.with_identity_stm(x)
    tf = rng.uniform(0.3, 0.9, n)
    for atol in (1e-12, 2.0 ** -310):
        r = batch.dop853_final(mu, y0, 0.0, tf, dim=dim, atol=atol, variant=variant,
                               max_steps=400)
        want, na, nr, st = oracle.batch_dop853_final(mu, y0, np.zeros(n), tf, atol=atol,
                                                     max_steps=400)
        assert np.array_equal(r.y.cpu().numpy(), want, equal_nan=True)
        assert np.array_equal(r.n_accepted.cpu().numpy(), na)
        assert np.array_equal(r.n_rejected.cpu().numpy(), nr)
        assert np.array_equal(r.status.cpu().numpy(), st)


@pytest.mark.parametrize("variant", ["plain", "wide", "pair", "persistent", "persistent_pair"])
def test_error_scales_at_their_bounds(gpu, oracle, variant):
    """STMs that start large enough for the error scale rtol |Phi| to lie on
    either side of 2^960, and small enough for entries below 2^-301."""
    n = 24
    rng = np.random.default_rng(3)
    y0 = W.with_identity_stm(W.planar_seeds(rng, n))
    size = 2.0 ** rng.permutation(np.array([0, 300, 500, 900, 998, 999, 1000, 1001, 1010, 1020,
                                            -200, -300, -301, -302, -500, -1000] + [0] * 8))
    y0[:, :36] *= size[:, None]
    y0[::3, 1] = 2.0 ** -310
    mu = np.full(n, MU)
    tf = rng.uniform(0.05, 0.4, n)
    r = batch.dop853_final(mu, y0, 0.0, tf, dim=42, variant=variant, max_steps=300)
    want, na, nr, st = oracle.batch_dop853_final(mu, y0, np.zeros(n), tf, max_steps=300)
    assert np.array_equal(r.y.cpu().numpy(), want, equal_nan=True)
    assert np.array_equal(r.n_accepted.cpu().numpy(), na)
    assert np.array_equal(r.n_rejected.cpu().numpy(), nr)
    assert np.array_equal(r.status.cpu().numpy(), st)


@pytest.mark.parametrize("n", [3, 4096, 4097])
def test_lane_groups_on_either_side_of_their_size_rule(gpu, n):
    """The 16- and 8-lane groups of the "wide" forms (up to 4,096 trajectories,
    more) against one trajectory per lane: fixed steps of every order, end
    states, grids and events, forward and backward, bit for bit."""
    rng = np.random.default_rng(n)
    y = W.planar_seeds(rng, n)
    y[:, 1] = rng.uniform(-0.02, 0.02, n)
    tf = rng.uniform(0.2, 1.5, n)

    def same(f):
        a, b = f("wide"), f("plain")
        for u, v in zip(a, b):
            assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())

    for fwd in (1, -1):
        for order in (4, 6, 8):
            same(lambda v: batch.rk_fixed(MU, y, 0.0, tf, 9, order=order, forward=fwd,
                                          return_derivatives=True, variant=v))
        kw = dict(forward=fwd, flip_indices=slice(0, 6) if fwd < 0 else None)
        same(lambda v: vars(batch.dop853_final(MU, y, 0.0, tf, variant=v, **kw)).values())
        same(lambda v: vars(batch.dop853_grid(MU, y, 0.0, tf, 7, variant=v, **kw)).values())
        same(lambda v: vars(batch.dop853_event(MU, y, 0.0, tf, variant=v, ev_index=1,
                                               **kw)).values())
        same(lambda v: vars(batch.dop853_event(MU, y, 0.0, tf, variant=v, ev_index=5,
                                               direction=1, **kw)).values())


@pytest.mark.parametrize("n,m", [(1, 2), (3, 130), (1024, 65), (1025, 65)])
def test_stm_grids_on_either_side_of_their_size_rule(gpu, oracle, n, m):
    """42-d grids up to 1,024 trajectories (two waves each) and beyond (lane
    groups): every point of sampled trajectories against the oracle, its end
    against the end-state kernels; more and fewer points than the 64 a wave
    forms at once, several in one step, shared output times, a zero span, an
    attempt limit, backward."""
    rng = np.random.default_rng(n)
    x = W.planar_seeds(rng, n)
    y0 = W.with_identity_stm(x)
    tf = rng.uniform(0.3, 1.2, n)
    tf[n // 2] = 0.0
    flip = slice(36, 42)
    t_eval = np.sort(rng.uniform(0.0, 0.7, m))
    t_eval[0] = 0.0
    some = sorted({0, n // 2, n - 1})
    for fwd in (1, -1):
        kw = dict(dim=42, forward=fwd, flip_indices=flip if fwd < 0 else None)
        g = batch.dop853_grid(MU, y0, 0.0, tf, m, **kw)
        e = batch.dop853_final(MU, y0, 0.0, tf, variant="plain", **kw)
        assert np.array_equal(g.states[:, -1].cpu().numpy(), e.y.cpu().numpy())
        assert np.array_equal(g.n_accepted.cpu().numpy(), e.n_accepted.cpu().numpy())
        shared = batch.dop853_grid(MU, y0, 0.0, 0.0, m, t_eval=t_eval, **kw)
        sys = oracle.System("cr3bp42", mu=MU, fwd=fwd, flip=flip if fwd < 0 else None)
        for i in some:
            want = np.repeat(y0[i][None], m, 0) if tf[i] == 0.0 else \
                oracle.compute_stm(MU, x[i], tf[i], steps=m, forward=fwd)[3]
            assert np.array_equal(g.states[i].cpu().numpy(), want)
            want = oracle.dop853(sys, y0[i], t_eval, rtol=1e-12, atol=1e-12, max_step=1e4)
            assert np.array_equal(shared.states[i].cpu().numpy(), want[0])
    cut = batch.dop853_grid(MU, y0, 0.0, tf, m, dim=42, max_steps=5)
    end = batch.dop853_final(MU, y0, 0.0, tf, dim=42, max_steps=5, variant="plain")
    assert np.array_equal(cut.status.cpu().numpy(), end.status.cpu().numpy())
    assert np.array_equal(cut.states[:, -1].cpu().numpy(), end.y.cpu().numpy())


@pytest.mark.parametrize("n", [4096, 4097])
def test_open_variant_on_either_side_of_its_rule(gpu, n):
    """dop853_final's 42-d default against the plain kernel, uneven spans with
    zero and reversed ones among them."""
    rng = np.random.default_rng(n)
    y0 = W.with_identity_stm(W.planar_seeds(rng, n))
    tf = rng.uniform(0.1, 1.0, n)
    tf[5], tf[6] = 0.0, -0.5
    a = batch.dop853_final(MU, y0, 0.0, tf, dim=42)
    b = batch.dop853_final(MU, y0, 0.0, tf, dim=42, variant="plain")
    for u, v in zip(vars(a).values(), vars(b).values()):
        assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())


@pytest.mark.parametrize("dim,variant", [(6, "plain"), (6, "wide"), (42, "plain"), (42, "wide"),
                                         (42, "pair"), (42, "persistent")])
@pytest.mark.parametrize("atol", [1e140, 1e152, 1e158, 1e200, 1e292])
def test_step_control_with_vanishing_errors(gpu, oracle, dim, variant, atol):
    """Error norms that underflow, or are exactly zero, as the controller's
    bases err and err_prev; large steps, the end's short ones."""
    n = 20
    rng = np.random.default_rng(4)
    x = W.planar_seeds(rng, n)
    y0 = x if dim == 6 else W.with_identity_stm(x)
    tf = rng.uniform(1e-4, 0.2, n)
    r = batch.dop853_final(MU, y0, 0.0, tf, dim=dim, atol=atol, variant=variant, max_step=0.01,
                           max_steps=300)
    want, na, nr, st = oracle.batch_dop853_final(np.full(n, MU), y0, np.zeros(n), tf, atol=atol,
                                                 max_step=0.01, max_steps=300)
    assert np.array_equal(r.y.cpu().numpy(), want)
    assert np.array_equal(r.n_accepted.cpu().numpy(), na)
    assert np.array_equal(r.n_rejected.cpu().numpy(), nr)
    assert np.array_equal(r.status.cpu().numpy(), st)


@pytest.mark.parametrize("n", [1, 6, 4097])
@pytest.mark.parametrize("m", [2, 15, 17, 129, 1500])
def test_grid_points_a_lane_each(gpu, n, m):
    """6-d grids of lane groups (up to 4,096 trajectories sixteen points at
    once) against one trajectory per lane: none, fewer and more points in a
    step than a group has lanes, output times that repeat or go back, a span of
    zero, an attempt limit, a step that covers points only at its end."""
    rng = np.random.default_rng(100 * n + m)
    y = W.planar_seeds(rng, n)
    y[:, 1:3] = rng.uniform(-0.02, 0.02, (n, 2))
    tf = rng.uniform(0.2, 1.5, n)
    tf[n // 2] = 0.0 if n > 1 else tf[0]
    t_eval = np.sort(rng.uniform(0.0, 0.7, m))
    t_eval[0] = 0.0
    again = t_eval.copy()
    again[m // 2:m // 2 + 3] = again[m // 2]
    back = t_eval.copy()
    back[m // 3:m // 3 + 2] = back[m // 3:m // 3 + 2][::-1]
    for fwd in (1, -1):
        for kw in (dict(), dict(max_steps=5), dict(max_step=0.05, max_steps=9), dict(t_eval=t_eval),
                   dict(t_eval=again), dict(t_eval=back)):
            a, b = (batch.dop853_grid(MU, y, 0.0, tf if "t_eval" not in kw else 0.0, m, variant=v,
                                      forward=fwd, **kw) for v in ("wide", "plain"))
            for u, v in zip(vars(a).values(), vars(b).values()):
                assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())
