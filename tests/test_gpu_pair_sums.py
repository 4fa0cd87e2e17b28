"""Rounding of the pair pass's sums (needs an MI355X).  Every 64 terms of an atom's sums are added in
FP32 and then folded into FP64, on the row side of a tile and on its column side, whatever the
tile's form.  With equal charges sum_j P q_j / f_ij is a sum of n like terms, whose FP32 runs of k terms
leave an error of about u sqrt(k / 3) each, n / k of them: u k / sqrt(3 n) of the whole.  A system's
first atoms are summed as rows, its last ones as columns, so equal runs on both sides scatter alike.
Each scatter is taken over 1 / 8 of the atoms (600 or more), which leaves 4 % on their ratio; runs of
128 terms on the column side make it 1.5 (the terms' own rounding is in both)."""
import numpy as np
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _pair_sums(prefactor, charge, born, pos, rows):
    """sum over j != i of P q_j / f_ij in FP64, from the FP32 values that the kernels read."""
    P, q, b = (np.asarray(v, dtype=np.float32).astype(np.float64) for v in (prefactor, charge, born))
    out = np.zeros(len(rows))
    for k in range(0, len(rows), 128):
        i = rows[k:k + 128]
        r2 = ((pos[i][:, None, :] - pos[None, :, :]) ** 2).sum(-1)
        bb = b[i][:, None] * b[None, :]
        term = q[None, :] / np.sqrt(r2 + bb * np.exp(-r2 / (4.0 * bb)))
        out[k:k + 128] = P * (term.sum(1) - term[np.arange(len(i)), i])
    return out


@pytest.mark.parametrize("n", [4800, 8900, 9025])  # one row block per wave; two, with even and odd blocks
def test_columns_round_like_rows(n):
    p = N.default_params(N.MODEL_GBSW)
    p.n_radial, p.n_lebedev = 12, 14
    s = S.globule(n, 5, iters=40)
    s.charge[:] = 1.0
    eng = N.Engine(p, s.charge, s.radius)
    dq = eng.execute_adjoint(s.pos)["dEdq"]
    born = eng.born_radii()
    eng.close()
    pairs = dq - p.prefactor * s.charge / born  # without the self term, which is added in FP64
    scatter = []
    for rows in (np.arange(n // 8), np.arange(n - n // 8, n)):
        scatter.append(float(np.std(pairs[rows] / _pair_sums(p.prefactor, s.charge, born, s.pos, rows) - 1.0)))
    print(f"[pair sums] N={n} relative scatter of the first atoms {scatter[0]:.2e}, of the last {scatter[1]:.2e}",
          flush=True)
    assert scatter[1] < 1.2 * scatter[0]
