"""gbi_execute_noalloc where cells hold more members than the lists keep (needs an MI355X): a small
cell_cap and dense systems.  Every member is laid out before a list is cut at the cap, so the
entries' capacity has to count them all; this entry point cannot grow it.  Against gbi_execute on
the same inputs at 1e-9 (the same kernels; FP64 summation order)."""
import numpy as np
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from test_zz_no_alloc import TOL, _allocating, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integral,n,scale,cap", [
    (N.INTEGRAL_GBMV2, 300, 1.0, 16),
    (N.INTEGRAL_GBMV1, 300, 1.0, 1),
    (N.INTEGRAL_GBSW, 400, 1.0, 3),
    (N.INTEGRAL_GBMV2, 900, 0.75, 64),
    (N.INTEGRAL_GBMV2, 1, 1.0, 64),
])
def test_lists_beyond_the_cap(integral, n, scale, cap):
    p = N.default_params(N.MODEL_GBMV, integral)
    p.cell_cap = cap
    s = S.globule(n, 51, iters=60)
    s.pos[:] = s.pos * scale
    print(f"[noalloc lists] integral {integral} N={n} scale {scale} cap {cap}", flush=True)
    e1, f1 = _noalloc(p, s)
    e0, f0 = _allocating(p, s)
    assert abs(e1 - e0) <= TOL * abs(e0)
    assert np.linalg.norm(f1 - f0) <= TOL * max(np.linalg.norm(f0), 1.0)
