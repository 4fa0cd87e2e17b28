"""Binning in batches of odd sizes (needs an MI355X): groups of two atoms end with their system, whose
last group may hold one, and the next system starts with other quadratures, grids and ways of
binning (bricks of fine cells; coarse cells; the GBSW forms).  Integrals and Born radii bitwise those of
single-system contexts, energies and forces against the FP64 oracle at the 1e-5 of the workload
specification."""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu

# (integral, atoms, radial, Lebedev, grid length)
BATCHES = [
    [(N.INTEGRAL_GBMV2, 5, 24, 50, 0.15), (N.INTEGRAL_GBMV2, 203, 24, 26, 0.15), (N.INTEGRAL_GBMV1, 3, 9, 14, 0.15)],
    [(N.INTEGRAL_GBMV1, 201, 10, 26, 0.15), (N.INTEGRAL_GBMV2, 7, 1, 6, 0.15), (N.INTEGRAL_GBMV2, 97, 40, 50, 0.12)],
    [(N.INTEGRAL_GBMV2, 151, 24, 38, 0.20), (N.INTEGRAL_GBMV1, 33, 24, 26, 0.30), (N.INTEGRAL_GBMV2, 65, 24, 26, 0.15)],
    [(N.INTEGRAL_GBSW, 51, 24, 38, 0.15), (N.INTEGRAL_GBMV2, 3, 24, 50, 0.15), (N.INTEGRAL_GBMV1, 129, 12, 38, 0.20)],
]


def _params(integral, radial, lebedev, grid):
    p = N.default_params(N.MODEL_GBMV, integral)
    p.n_radial, p.n_lebedev, p.grid_length = radial, lebedev, grid
    return p


@pytest.mark.parametrize("which", range(len(BATCHES)))
def test_batch_bins_like_single_systems(which):
    kinds = BATCHES[which]
    systems = [S.globule(k[1], 70 + k[1]) for k in kinds]
    params = [_params(k[0], *k[2:]) for k in kinds]
    print(f"[bins batch] {kinds}", flush=True)
    batch = N.Engine.batch(params, [s.charge for s in systems], [s.radius for s in systems])
    e, f = batch.execute(np.concatenate([s.pos for s in systems]))
    e2, f2 = batch.execute(np.concatenate([s.pos for s in systems]))
    integrals, born, at = batch.integrals(), batch.born_radii(), batch.offsets
    batch.close()
    assert np.array_equal(e2, e) and np.array_equal(f2, f)
    for k, (p, s) in enumerate(zip(params, systems)):
        cut = slice(at[k], at[k + 1])
        eng = N.Engine(p, s.charge, s.radius)
        eng.execute(s.pos)
        assert np.array_equal(integrals[:, cut], eng.integrals())
        assert np.array_equal(born[cut], eng.born_radii())
        eng.close()
        ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), s.pos, s.charge, s.radius)
        assert rel_err(e[k], ref.energy) < 1e-5
        assert rel_rms(f[cut], ref.forces) < 1e-5
