"""Periodic cutoff systems whose atoms move between evaluations of one context, directly and by graph
replay (needs an MI355X): the pair tiles write only the partial sums of blocks in reach, and blocks come
into and out of reach through the box's faces as halves of the liquid shift.  Against the FP64 oracle
at the 1e-5 of the workload specification; the first positions again give the first results bit for bit."""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params, rel_err, rel_rms

pytestmark = pytest.mark.gpu
BOX = (2.6, 2.7, 3.0)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("model,integral", [(N.MODEL_GBSW, N.INTEGRAL_GBSW), (N.MODEL_GBMV, N.INTEGRAL_GBMV2)])
def test_blocks_move_through_the_box(model, integral, graph):
    p = N.default_params(model, integral)
    p.n_radial, p.n_lebedev = 12, 14
    p.nonbonded_method, p.cutoff = N.CUTOFF_PERIODIC, 0.7
    s = S.liquid(BOX, 4, density=45.0, iters=60)
    half = np.arange(s.n) >= s.n // 2
    frames = [s.pos]
    for shift in ((0.4, 0.0, 0.9), (0.0, 1.3, -1.1)):
        x = s.pos.copy()
        x[half] += shift
        frames.append(x)
    print(f"[periodic moves] model {model} N={s.n} graph {graph}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)
    eng.set_periodic_box(BOX)
    eng.set_graph(graph)
    first = eng.execute(frames[0])
    for x in (frames[1], frames[0], frames[2]):
        e, f = eng.execute(x)
        ref = O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1), box=BOX), x, s.charge, s.radius)
        assert rel_err(e, ref.energy) < 1e-5
        assert rel_rms(f, ref.forces) < 1e-5
    again = eng.execute(frames[0])
    eng.close()
    assert again[0] == first[0] and np.array_equal(again[1], first[1])
