"""GBSW cells that atoms leave between evaluations of one context (needs an MI355X): two halves of a
molecule apart by many empty cells, together, and apart along another axis.  An empty cell's masks must
say V = 1 whatever an earlier evaluation left there.  Against the FP64 oracle at the 1e-5 of the
workload specification; the first positions again give the first results bit for bit."""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", [N.MODEL_GBSW, N.MODEL_GBMV])
def test_cells_left_by_their_atoms(model):
    p = N.default_params(model, N.INTEGRAL_GBSW)
    s = S.globule(240, 17)
    half = s.pos[:, 0] > np.median(s.pos[:, 0])
    frames = [s.pos.copy() for _ in range(3)]
    frames[0][half, 0] += 4.0
    frames[2][half, 1] += 3.0
    eng = N.Engine(p, s.charge, s.radius)
    first = eng.execute(frames[0])
    for x in (*frames, frames[1]):
        print(f"[gbsw sparse] model {model} extent {np.ptp(x, axis=0).round(1)}", flush=True)
        e, f = eng.execute(x)
        ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), x, s.charge, s.radius)
        assert rel_err(e, ref.energy) < 1e-5
        assert rel_rms(f, ref.forces) < 1e-5
    again = eng.execute(frames[0])
    eng.close()
    assert again[0] == first[0] and np.array_equal(again[1], first[1])
