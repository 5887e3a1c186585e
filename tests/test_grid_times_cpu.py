"""CPU: the ends of explicit output times are the first and last of the times
as converted, whatever sequence the caller holds them in."""
import collections
import ctypes as C

import numpy as np
import pandas as pd
import pytest
import torch

from hiten_amd import _lib, batch

T = np.array([0.25, 0.5, 1.0, 1.75])


class _Library:
    """Takes hh_dop853_grid's place and keeps the times it is given."""

    def hh_dop853_grid(self, n, dim, mu, t0, tf, m, te, *rest):
        row = lambda p, k: np.ctypeslib.as_array((C.c_double * k).from_address(p)).copy()
        self.got = row(t0, n), row(tf, n), row(te, m)
        return 0


@pytest.mark.parametrize("times", [
    T, list(T), tuple(T), collections.deque(T), torch.tensor(T), T.astype(np.float32),
    torch.tensor(T, dtype=torch.float16), [str(t) for t in T], list(map(np.array, T)),
    pd.Series(T), pd.Series(T, index=[3, 2, 1, 0]), pd.Series(T, index=[5, 6, 7, 8]),
    pd.Series(T, index=list("abcd")), pd.Index(T)], ids=lambda t: type(t).__name__)
def test_ends_of_explicit_times(monkeypatch, times):
    lib = _Library()
    monkeypatch.setattr(_lib, "load", lambda *a, **k: lib)
    monkeypatch.setattr(batch, "_device", lambda: torch.device("cpu"))
    monkeypatch.setattr(batch, "_launch_stream", lambda *a: 0)
    batch.dop853_grid(0.01, np.zeros((3, 6)), None, None, 0, t_eval=times)
    t0, tf, te = lib.got
    assert (t0 == T[0]).all() and (tf == T[-1]).all() and np.array_equal(te, T)


def test_no_times_are_refused(monkeypatch):
    monkeypatch.setattr(_lib, "load", lambda *a, **k: _Library())
    monkeypatch.setattr(batch, "_device", lambda: torch.device("cpu"))
    with pytest.raises(IndexError):
        batch.dop853_grid(0.01, np.zeros((3, 6)), None, None, 0, t_eval=[])
