"""gbi_get_stats of GBSW, GBMV and mixed contexts (needs an MI355X): bytes of a binned point's slot by the
kind of system (GBSW points are not binned), and counts that add up over a batch."""
import numpy as np
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


def test_slot_bytes_and_counts():
    params = [N.default_params(N.MODEL_GBSW), N.default_params(N.MODEL_GBMV, N.INTEGRAL_GBMV2)]
    systems = [S.globule(90, 1), S.globule(210, 2)]
    got = []
    for p, s in zip(params, systems):
        eng = N.Engine(p, s.charge, s.radius)
        eng.execute(s.pos)
        got.append(eng.stats())
        eng.close()
    eng = N.Engine.batch(params, [s.charge for s in systems], [s.radius for s in systems])
    eng.execute(np.concatenate([s.pos for s in systems]))
    both = eng.stats()
    eng.close()
    assert got[0]["slot_bytes"] == 0.0 and got[1]["slot_bytes"] == 4.0
    assert both["slot_bytes"] == pytest.approx(4.0 * 210 / 300)
    for key in ("n_points", "n_vol_pairs", "n_entries", "n_active", "n_frc_pairs"):
        assert got[0][key] > 0 and got[1][key] > 0
        assert both[key] == got[0][key] + got[1][key], key
