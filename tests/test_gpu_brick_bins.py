"""Binning by bricks, a few atoms per workgroup, at the sizes where it can go wrong (needs an
MI355X): a last group with fewer atoms, fewer points in a group than a workgroup's threads, the
most points that its table is sized for, and groups of a batch, which never span two systems.
Against the FP64 oracle at the 1e-5 of the workload specification; alone and in a batch bitwise.
"""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu


def _params(itype, radial, lebedev):
    p = N.default_params(N.MODEL_GBMV, itype)
    p.n_radial, p.n_lebedev = radial, lebedev
    return p


@pytest.mark.parametrize("n,itype,radial,lebedev", [
    (3, N.INTEGRAL_GBMV2, 24, 50),
    (5, N.INTEGRAL_GBMV2, 1, 6),      # 6 points per atom
    (101, N.INTEGRAL_GBMV1, 10, 26),  # 260: groups of about a workgroup's threads
    (203, N.INTEGRAL_GBMV2, 40, 50),  # 2,000 points per atom
    (1001, N.INTEGRAL_GBMV2, 24, 38),
])
def test_groups_match_oracle(n, itype, radial, lebedev):
    p = _params(itype, radial, lebedev)
    s = S.globule(n, 13)
    print(f"[brick bins] N={n} type {itype} {radial}x{lebedev}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)
    e, f = eng.execute(s.pos)
    e2, f2 = eng.execute(s.pos)
    eng.close()
    ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), s.pos, s.charge, s.radius)
    assert e2 == e and np.array_equal(f2, f)
    assert rel_err(e, ref.energy) < 1e-5
    assert rel_rms(f, ref.forces) < 1e-5
