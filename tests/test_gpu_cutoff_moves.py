"""Cutoff systems whose atoms move between evaluations of one context (needs an MI355X): the pair
tiles write the partial sums of the blocks in reach only, and the next pass reads no others, so
sums of an earlier evaluation must never come back.  Two halves are drawn apart beyond the
cutoff and pushed together again; sizes at the edges of 64-atom blocks and of the two tile forms.
Against the FP64 oracle at the 1e-5 of the workload specification; the first
positions again give the first results bit for bit."""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cutoff", [(64, 0.5), (129, 0.6), (700, 0.8), (3073, 1.0), (3200, 1.6)])
@pytest.mark.parametrize("adjoint", [False, True])
def test_partials_of_other_positions_do_not_return(n, cutoff, adjoint):
    p = N.default_params(N.MODEL_GBSW)
    p.nonbonded_method, p.cutoff = N.CUTOFF_NON_PERIODIC, cutoff
    s = S.globule(n, 31)
    apart = s.pos.copy()
    apart[s.pos[:, 0] > np.median(s.pos[:, 0]), 0] += 2.0
    print(f"[cutoff moves] N={n} cutoff {cutoff} adjoint {adjoint}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)

    def run(pos):
        if adjoint:
            a = eng.execute_adjoint(pos)
            return a["energy"], a["forces"]
        return eng.execute(pos)

    first = run(s.pos)
    for pos in (apart, s.pos, apart):
        e, f = run(pos)
        ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), pos, s.charge, s.radius)
        assert rel_err(float(np.ravel(e)[0]), ref.energy) < 1e-5
        assert rel_rms(np.reshape(f, pos.shape), ref.forces) < 1e-5
    again = run(s.pos)
    assert np.array_equal(np.asarray(again[0]), np.asarray(first[0])) and np.array_equal(again[1], first[1])
    eng.close()
