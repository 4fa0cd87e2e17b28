"""The batch-wide flags of k_bbox (needs an MI355X): the workgroup that finishes the last system
writes them, whichever system raised one and however many slices (1,024 atoms) its bounding box
takes, and the counts behind that are back at zero for the next evaluation.  An evaluation
with a non-finite position on the device is refused; the next one gives the first one's results bit
for bit."""
import numpy as np
import pytest
import torch  # before the library loads the HIP runtime (device-resident positions below)

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,bad", [
    ((40,), 0),
    ((2300,), 0),            # three slices
    ((40, 1100, 65), 0),
    ((40, 1100, 65), 1),     # the system of two slices
    ((40, 1100, 65), 2),
    ((12,) * 70, 69),        # more systems than a wave
])
def test_one_system_flags_the_batch(sizes, bad):
    systems = [S.globule(n, 20 + k) for k, n in enumerate(sizes)]
    params = [N.default_params(N.MODEL_GBSW) for _ in sizes]
    eng = N.Engine.batch(params, [s.charge for s in systems], [s.radius for s in systems])
    pos = np.concatenate([s.pos for s in systems])
    print(f"[batch flags] {len(sizes)} systems, {pos.shape[0]} atoms, bad system {bad}", flush=True)
    e, f = eng.execute(pos)
    wrong = pos.copy()
    wrong[sum(sizes[:bad]) + sizes[bad] - 1, 2] = np.nan
    d = torch.tensor(wrong, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):
        eng.set_positions(d.data_ptr(), on_device=True)
        eng.compute()
        with pytest.raises(N.GbiError) as ex:
            eng.synchronize()
        assert ex.value.status == 7
        e2, f2 = eng.execute(pos)
        assert np.array_equal(np.asarray(e2), np.asarray(e)) and np.array_equal(f2, f)
    eng.close()
