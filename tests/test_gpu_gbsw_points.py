"""k_gbsw_points at the sizes where it can go wrong (needs an MI355X): fewer points per atom
than a workgroup's threads and many more (its queue in several rounds, the largest quadrature),
lists at and beyond 63 atoms (whole-list scan instead of the sub-cells' bits), sub-cells near
the atoms' size and far above it, the unbounded brute cell, and slots that overflow and grow.
Energy, forces and Born radii against the FP64 oracle at the 1e-5 of the workload specification.
"""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu


def _close_pack(n, spacing, seed):
    """A lattice denser than the slots are sized for: 0.15 nm spacing is 300 atoms/nm^3."""
    k = int(np.ceil(n ** (1 / 3)))
    idx = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    rng = np.random.default_rng(seed)
    pos = idx * spacing + rng.uniform(-0.01, 0.01, idx.shape)
    q = rng.uniform(-0.8, 0.8, n)
    return S.System(pos, q - q.mean(), np.full(n, 0.04))


@pytest.mark.parametrize("n,radial,lebedev,tight,brute,dense", [
    (2, 24, 38, 0.20, False, False),
    (97, 1, 6, 0.20, False, False),      # 6 points per atom
    (301, 10, 26, 0.20, False, False),   # 260: one more round than 256
    (257, 40, 50, 0.20, False, False),   # 2,000 points
    (300, 24, 38, 0.05, False, False),   # sub-cells of 0.0125 nm
    (500, 24, 38, 0.40, False, False),   # lists around 63 atoms
    (700, 24, 38, 0.90, False, False),   # scans
    (130, 24, 38, 0.20, True, False),
    (900, 24, 50, 0.25, False, True),    # small, crowded spheres: most points of a cell are active
])
def test_points_match_oracle(n, radial, lebedev, tight, brute, dense):
    p = N.default_params(N.MODEL_GBSW)
    p.n_radial, p.n_lebedev, p.tight_grid_length = radial, lebedev, tight
    if brute:
        p.lookup_policy = N.LOOKUP_BRUTE
    s = _close_pack(n, 0.15, 3) if dense else S.globule(n, 11)
    print(f"[gbsw points] N={n} {radial}x{lebedev} tight {tight} brute {brute} dense {dense}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)
    e, f = eng.execute(s.pos)
    e2, f2 = eng.execute(s.pos)
    born = eng.born_radii()
    eng.close()
    ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1)), s.pos, s.charge, s.radius)
    assert e2 == e and np.array_equal(f2, f)  # slots fill in any order; the results do not depend on it
    assert float(np.max(np.abs(born - ref.born) / ref.born)) < 1e-5
    assert rel_err(e, ref.energy) < 1e-5
    assert rel_rms(f, ref.forces) < 1e-5
