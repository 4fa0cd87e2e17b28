"""Sparse and elongated GBSW systems in gbi_execute_noalloc: many cells for few points, up to what its
256 MiB scratch array holds.  The size check (no GPU needed: it comes before the device is looked
for) accepts each; on an MI355X the results are those of gbi_execute at 1e-9 (the same kernels)."""
import ctypes

import numpy as np
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

CASES = [("gbsw", 100, 5.0), ("gbsw", 300, 4.0), ("gbsw", 600, 3.0), ("gbsw", 2000, 1.0),
         ("gbmv", 100, 5.0), ("gbmv", 300, 4.0), ("gbmv", 1500, 2.0), ("brute", 40, 30.0)]
INVALID_ARGUMENT = 1


def _case(kind, n, apart):
    p = N.default_params(N.MODEL_GBMV, N.INTEGRAL_GBSW) if kind == "gbmv" else N.default_params(N.MODEL_GBSW)
    if kind == "brute":
        p.lookup_policy = N.LOOKUP_BRUTE
    s = S.globule(n, 71)
    pos = s.pos.copy()
    pos[pos[:, 0] > np.median(pos[:, 0])] += apart  # two halves drawn apart along the diagonal
    return p, s, pos


def _noalloc(p, s, pos):
    lib = N.load()
    e, f = np.zeros(1), np.zeros((s.n, 3))
    st = lib.gbi_execute_noalloc(s.n, N._dp(s.charge), N._dp(s.radius), ctypes.byref(p), N._dp(pos), 1, 1, N._dp(e),
                                 N._dp(f), None)
    return st, lib.gbi_last_error(), float(e[0]), f


@pytest.mark.parametrize("kind,n,apart", CASES)
def test_size_check_accepts(kind, n, apart):
    st, message, _, _ = _noalloc(*_case(kind, n, apart))
    assert st != INVALID_ARGUMENT, message


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,apart", CASES)
def test_results(kind, n, apart):
    p, s, pos = _case(kind, n, apart)
    print(f"[noalloc sizes] {kind} N={n} apart {apart}", flush=True)
    st, message, e1, f1 = _noalloc(p, s, pos)
    assert st == N.GBI_OK, message
    eng = N.Engine(p, s.charge, s.radius)
    e0, f0 = eng.execute(pos)
    eng.close()
    assert abs(e1 - e0) < 1e-9 * abs(e0)
    assert np.linalg.norm(f1 - f0) < 1e-9 * np.linalg.norm(f0)
