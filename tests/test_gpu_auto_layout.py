"""GPU: end states with the layout left open do not depend on the process-wide
scheduling settings, on either side of the layout's size rule."""

import numpy as np
import pytest
import torch

from hiten_amd import _lib, batch, workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 4097])
def test_open_layout_gives_the_same_bits_under_every_setting(gpu, n):
    rng = np.random.default_rng(n)
    y = W.with_identity_stm(W.planar_seeds(rng, n))
    tf = rng.uniform(0.05, 0.5, n)
    want = batch.dop853_final(W.MU_EM, y, 0.0, tf, dim=42, variant="plain")
    saved = _lib.get_tuning()
    try:
        for kw in (dict(), dict(heavy_projected=3, min_age=1),
                   dict(heavy_projected=0, min_age=1000)):
            _lib.set_tuning(**{**saved, **kw})
            got = batch.dop853_final(W.MU_EM, y, 0.0, tf, dim=42)
            for g, e in zip(vars(got).values(), vars(want).values()):
                assert torch.equal(g, e)
    finally:
        _lib.set_tuning(**saved)
