"""A caller's own graph: gbi_set_positions (device) and gbi_compute captured on the caller's stream
and replayed with other positions in the same buffer (needs an MI355X).  After every replay, with
eager work and a synchronization of the caller's between them, the energy, forces and Born radii
read back are those of an eager evaluation of the same positions, bit for bit."""
import numpy as np
import pytest
import torch

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,integral,cutoff", [
    (N.MODEL_GBSW, N.INTEGRAL_GBSW, None),
    (N.MODEL_GBSW, N.INTEGRAL_GBSW, 0.8),
    (N.MODEL_GBMV, N.INTEGRAL_GBMV2, None),
])
def test_replays_read_back_fresh(model, integral, cutoff):
    p = N.default_params(model, integral)
    if cutoff:
        p.nonbonded_method, p.cutoff = N.CUTOFF_NON_PERIODIC, cutoff
    s = S.globule(300, 41)
    frames = [s.pos] + [c.pos for c in S.conformations(s, 3, 42)]
    print(f"[caller graph] model {model} integral {integral} cutoff {cutoff}", flush=True)
    ref = N.Engine(p, s.charge, s.radius)
    ref.execute(s.pos)  # buffers and, with a cutoff, the pair order from the same first positions
    want = []
    for x in frames:
        e, f = ref.execute(x)
        want.append((e, f, ref.born_radii()))
    ref.close()

    eng = N.Engine(p, s.charge, s.radius)
    stream = torch.cuda.Stream()
    eng.set_stream(stream.cuda_stream)
    x = torch.from_numpy(s.pos.copy()).cuda()
    torch.cuda.synchronize()
    eng.set_positions(x.data_ptr(), on_device=True)
    eng.compute()
    eng.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        eng.set_positions(x.data_ptr(), on_device=True)
        eng.compute()
    for k in (1, 2, 0, 3, 2):
        x.copy_(torch.from_numpy(frames[k]))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        stream.synchronize()
        e, f, born = want[k]
        assert eng.energy() == e
        assert np.array_equal(eng.forces(), f)
        assert np.array_equal(eng.born_radii(), born)
        eng.synchronize()
        assert eng.energy() == e
    eng.close()
