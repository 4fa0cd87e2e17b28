"""GBSW with wide switching shells, whose points are binned into cells (half-widths above 0.09 nm; needs
an MI355X): at the line between the two forms, far beyond it, with the truncated chain rule of a
cutoff, periodic, on both grids, with quadratures of no multiple of four, lists longer than a staged
chunk, in batches beside the other kinds, in gbi_execute_noalloc, and when gbi_update_constants
moves the width across the line.  Against the FP64 oracle at the 1e-5 of the workload specification."""
import os

import numpy as np
import pytest

import oracle as O
from openmmcustomgbintegralforce_amd import _native as N
from openmmcustomgbintegralforce_amd import synthetic as S

from common import oracle_params
from test_zz_no_alloc import TOL, _noalloc

pytestmark = pytest.mark.gpu
LINE = 0.09
BOX = (2.4, 2.5, 2.6)


def _params(model, w, method=N.NO_CUTOFF, cutoff=0.8, radial=24, lebedev=38):
    p = N.default_params(model, N.INTEGRAL_GBSW)
    p.sw, p.nonbonded_method, p.cutoff, p.n_radial, p.n_lebedev = w, method, cutoff, radial, lebedev
    return p


def _system(n, method, scale=1.0):
    s = S.liquid(BOX, 8, density=n / float(np.prod(BOX)), iters=40) if method == N.CUTOFF_PERIODIC else S.globule(n, 9)
    s.pos[:] = s.pos * scale
    return s


def _oracle(p, s, method):
    return O.compute(oracle_params(p, nthreads=min(16, os.cpu_count() or 1),
                                   box=BOX if method == N.CUTOFF_PERIODIC else None), s.pos, s.charge, s.radius)


@pytest.mark.parametrize("model,w,method,n,radial,lebedev,scale", [
    (N.MODEL_GBSW, LINE, N.NO_CUTOFF, 203, 24, 38, 1.0),
    (N.MODEL_GBSW, LINE + 1e-6, N.NO_CUTOFF, 203, 24, 38, 1.0),
    (N.MODEL_GBSW, 0.2, N.NO_CUTOFF, 301, 9, 14, 1.0),   # 126 points per atom
    (N.MODEL_GBSW, 0.5, N.NO_CUTOFF, 500, 10, 14, 0.6),  # lists beyond 256 atoms
    (N.MODEL_GBSW, 0.12, N.CUTOFF_NON_PERIODIC, 203, 24, 38, 1.0),
    (N.MODEL_GBSW, 0.12, N.CUTOFF_PERIODIC, 700, 12, 26, 1.0),
    (N.MODEL_GBMV, 0.1, N.NO_CUTOFF, 301, 24, 38, 1.0),
    (N.MODEL_GBMV, 0.2, N.CUTOFF_NON_PERIODIC, 203, 9, 14, 1.0),
    (N.MODEL_GBMV, 0.1, N.CUTOFF_PERIODIC, 700, 12, 26, 1.0),
    (N.MODEL_GBSW, 0.2, N.NO_CUTOFF, 1, 24, 38, 1.0),
])
def test_wide_shells_match_oracle(model, w, method, n, radial, lebedev, scale):
    p, s = _params(model, w, method, radial=radial, lebedev=lebedev), _system(n, method, scale)
    print(f"[gbsw wide] model {model} w {w} method {method} N={s.n} {radial}x{lebedev}", flush=True)
    eng = N.Engine(p, s.charge, s.radius)
    if method == N.CUTOFF_PERIODIC:
        eng.set_periodic_box(BOX)
    e, f = eng.execute(s.pos)
    again = eng.execute(s.pos)
    adj = eng.execute_adjoint(s.pos)
    eng.close()
    ref = _oracle(p, s, method)
    assert again[0] == e and np.array_equal(again[1], f)
    assert adj["energy"] == e and np.array_equal(adj["forces"], f)
    # (a single atom of the globule has no charge: zero energy and forces)
    assert abs(e - ref.energy) <= 1e-5 * abs(ref.energy)
    assert np.linalg.norm(f - ref.forces) <= 1e-5 * np.linalg.norm(ref.forces)
    assert abs(float(np.dot(s.charge, adj["dEdq"])) - 2.0 * e) <= 2e-5 * abs(e)  # E is quadratic in the charges


def test_adjoint_of_wide_shells():
    """Central differences of the oracle's energy in w, rscale and a radius (the bound of the narrow
    form's test: 1e-3 of the derivative)."""
    p, s = _params(N.MODEL_GBSW, 0.12), _system(150, N.NO_CUTOFF)
    eng = N.Engine(p, s.charge, s.radius)
    adj = eng.execute_adjoint(s.pos)
    eng.close()

    def energy(radius=s.radius, **const):
        q = _params(N.MODEL_GBSW, 0.12)
        for k, v in const.items():
            setattr(q, k, v)
        return O.compute(oracle_params(q, nthreads=min(16, os.cpu_count() or 1)), s.pos, s.charge, radius).energy

    h = 1e-5
    for name, at in (("sw", p.sw), ("rscale", p.rscale)):
        fd = (energy(**{name: at + h}) - energy(**{name: at - h})) / (2 * h)
        assert abs(adj["dEdtheta"][name] - fd) < 1e-3 * abs(fd), name
    j = int(np.argmax(np.abs(adj["dEdR"])))
    step = np.zeros(s.n)
    step[j] = h
    fd = (energy(s.radius + step) - energy(s.radius - step)) / (2 * h)
    assert abs(adj["dEdR"][j] - fd) < 1e-3 * abs(fd)


@pytest.mark.parametrize("model", [N.MODEL_GBSW, N.MODEL_GBMV])
def test_constants_across_the_line(model):
    s = _system(260, N.NO_CUTOFF)
    p = _params(model, 0.03)
    eng = N.Engine(p, s.charge, s.radius)
    eng.set_graph(True)
    for w in (0.03, 0.15, 0.05, 0.3, 0.03):
        p.sw = w
        eng.update_constants(p)
        got = eng.execute_adjoint(s.pos)
        fresh = N.Engine(p, s.charge, s.radius)
        want = fresh.execute_adjoint(s.pos)
        fresh.close()
        assert got["energy"] == want["energy"] and np.array_equal(got["forces"], want["forces"]), w
        assert np.array_equal(got["dEdR"], want["dEdR"]) and got["dEdtheta"] == want["dEdtheta"], w
    eng.close()


def test_beside_the_other_kinds():
    systems = [S.globule(n, 30 + n) for n in (97, 200, 33, 64)]
    params = [_params(N.MODEL_GBSW, 0.12), N.default_params(N.MODEL_GBMV, N.INTEGRAL_GBMV2),
              _params(N.MODEL_GBSW, 0.03), _params(N.MODEL_GBMV, 0.2)]
    batch = N.Engine.batch(params, [s.charge for s in systems], [s.radius for s in systems])
    e, f = batch.execute(np.concatenate([s.pos for s in systems]))
    integrals, at = batch.integrals(), batch.offsets
    batch.close()
    for k, (p, s) in enumerate(zip(params, systems)):
        eng = N.Engine(p, s.charge, s.radius)
        e0, f0 = eng.execute(s.pos)
        assert np.array_equal(integrals[:, at[k]:at[k + 1]], eng.integrals())
        eng.close()
        assert abs(e[k] - e0) <= 1e-12 * abs(e0)
        assert np.linalg.norm(f[at[k]:at[k + 1]] - f0) <= 1e-7 * np.linalg.norm(f0)


@pytest.mark.parametrize("model", [N.MODEL_GBSW, N.MODEL_GBMV])
def test_without_allocations(model):
    p, s = _params(model, 0.15), _system(300, N.NO_CUTOFF)
    e1, f1 = _noalloc(p, s)
    eng = N.Engine(p, s.charge, s.radius)
    e0, f0 = eng.execute(s.pos)
    eng.close()
    assert abs(e1 - e0) < TOL * abs(e0) and np.linalg.norm(f1 - f0) < TOL * np.linalg.norm(f0)
