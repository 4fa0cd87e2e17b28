"""Batches that mix all-pairs, cutoff and excluded-pair systems (needs an MI355X).  The form of a
system's pair tiles goes by the system alone, so its FP32 sums are grouped as when it is alone, and
only FP64 sums may take another order (the length of a tile follows the batch): integrals bitwise,
dE/dq to 1e-12, whatever its neighbours are.  Atoms move between evaluations, so that the partial
sums that a cutoff tile leaves out (and those of an earlier evaluation in their place) would show;
directly and by graph replay."""
import numpy as np
import pytest

from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

pytestmark = pytest.mark.gpu


def _params(kind, cutoff):
    p = N.default_params(N.MODEL_GBSW) if kind == "gbsw" else N.default_params(N.MODEL_GBMV, N.INTEGRAL_GBMV2)
    p.n_radial, p.n_lebedev = 10, 14
    if cutoff:
        p.nonbonded_method, p.cutoff = N.CUTOFF_NON_PERIODIC, cutoff
    return p


def _evaluate(eng, pos):
    a = eng.execute_adjoint(pos)
    return {"E": np.atleast_1d(a["energy"]), "F": a["forces"], "dq": a["dEdq"], "I": eng.integrals()}


# (model, atoms, cutoff, excluded pairs)
BIG = ("gbsw", 8900, None, None)
MIXES = [
    [BIG, ("gbsw", 300, 0.6, None)],
    [("gbmv", 129, None, [[0, 128], [3, 4]]), BIG],
    [("gbmv", 3200, 0.9, None), ("gbsw", 700, 0.8, None), BIG, ("gbmv", 65, None, [[0, 64]])],
]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("mix", range(len(MIXES)))
def test_a_system_has_the_sums_it_has_alone(mix, graph):
    kinds = MIXES[mix]
    systems = [S.globule(n, 60 + k, iters=40) for k, (_, n, _, _) in enumerate(kinds)]
    params = [_params(m, c) for m, _, c, _ in kinds]
    print(f"[mixed tiles] {[k[:3] for k in kinds]} graph {graph}", flush=True)
    frames = [[s.pos for s in systems], [], [s.pos for s in systems]]
    for s in systems:  # drawn apart along x beyond every cutoff
        x = s.pos.copy()
        x[s.pos[:, 0] > np.median(s.pos[:, 0]), 0] += 2.0
        frames[1].append(x)

    batch = N.Engine.batch(params, [s.charge for s in systems], [s.radius for s in systems])
    batch.set_graph(graph)
    alone = [N.Engine(p, s.charge, s.radius) for p, s in zip(params, systems)]
    for k, (_, _, _, excl) in enumerate(kinds):
        if excl:
            batch.set_exclusions(excl, system=k)
            alone[k].set_exclusions(excl)
    at = batch.offsets
    for frame in frames:
        got = _evaluate(batch, np.concatenate(frame))
        for k, eng in enumerate(alone):
            want, cut = _evaluate(eng, frame[k]), slice(at[k], at[k + 1])
            assert np.array_equal(got["I"][:, cut], want["I"])
            assert np.abs(got["dq"][cut] - want["dq"]).max() <= 1e-12 * np.abs(want["dq"]).max()
            assert abs(got["E"][k] - want["E"][0]) <= 1e-12 * abs(want["E"][0])
            # FP32 chain-rule factors of FP64 sums in another order, quantised to 2^-24
            assert np.linalg.norm(got["F"][cut] - want["F"]) <= 1e-7 * np.linalg.norm(want["F"])
    for eng in (batch, *alone):
        eng.close()
