"""Engine.set_tuning changes only what it is given (needs an MI355X): its default workgroups per CU are
the library's own."""
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


def test_set_tuning_keeps_the_library_default():
    s = S.globule(20, 3)
    eng = N.Engine(N.default_params(N.MODEL_GBSW), s.charge, s.radius)
    before = eng.tuning()
    eng.set_tuning(pair_columns=128)
    after = eng.tuning()
    eng.close()
    assert after["pair_columns"] == 128
    assert after["blocks_per_cu"] == before["blocks_per_cu"]
