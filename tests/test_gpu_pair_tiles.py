"""The pair pass's tile forms at the sizes where they change (needs an MI355X): 4 waves per tile up
to 3,072 atoms, one row block per wave above, two from 8,897; a last block of one atom, an odd
last row block, a cutoff (no two-row tiles), the adjoint, and exclusions set on a context whose
tiles have two rows.  A coarse quadrature keeps the oracle to the pair terms.
"""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu


def _params(cutoff=None, model=N.MODEL_GBSW):
    p = N.default_params(model, N.INTEGRAL_GBSW)
    p.n_radial, p.n_lebedev = 12, 14
    if cutoff:
        p.nonbonded_method, p.cutoff = N.CUTOFF_NON_PERIODIC, cutoff
    return p


@pytest.mark.parametrize("n,cutoff", [(63, None), (64, None), (65, None), (129, 0.7), (3072, None), (3073, None),
                                      (3073, 1.1), (8896, None), (8897, None), (9024, None), (9025, 1.1)])
def test_tiles_match_oracle(n, cutoff):
    p, s = _params(cutoff), S.globule(n, 5, iters=40)
    print(f"[tiles] N={n} cutoff {cutoff}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)
    e, f = eng.execute(s.pos)
    adj = eng.execute_adjoint(s.pos)
    eng.close()
    ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), s.pos, s.charge, s.radius)
    assert rel_err(e, ref.energy) < 1e-5
    assert rel_rms(f, ref.forces) < 1e-5
    assert adj["energy"] == e and np.array_equal(adj["forces"], f)
    assert rel_err(float(np.dot(s.charge, adj["dEdq"])), 2.0 * e) < 1e-5  # E is quadratic in the charges


def test_exclusions_on_two_row_tiles():
    p, s = _params(model=N.MODEL_GBMV), S.globule(9000, 6, iters=40)
    eng = N.Engine(p, s.charge, s.radius)
    e0, f0 = eng.execute(s.pos)
    pairs = np.array([[0, 1], [0, 8999], [63, 64], [4000, 4100]], dtype=np.int32)
    eng.set_exclusions(pairs)
    e1, _ = eng.execute(s.pos)
    born = eng.born_radii()
    eng.set_exclusions(np.zeros((0, 2), dtype=np.int32))
    e2, f2 = eng.execute(s.pos)
    eng.close()
    d = np.linalg.norm(s.pos[pairs[:, 0]] - s.pos[pairs[:, 1]], axis=1)
    bb = born[pairs[:, 0]] * born[pairs[:, 1]]
    pair = p.prefactor * s.charge[pairs[:, 0]] * s.charge[pairs[:, 1]] / np.sqrt(d * d + bb * np.exp(-d * d / (4 * bb)))
    # the energy's own FP32 rounding (3e-8 of it) against the excluded terms
    assert abs((e0 - e1) - pair.sum()) < 1e-6 * abs(e0)
    assert e2 == e0 and np.array_equal(f2, f0)
