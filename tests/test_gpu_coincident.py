"""Particles at exactly one point (GPU): a neighbour at distance 0 has F(0), so
density, h and sound speed are the oracle's in every search that can meet it,
the first pass, the walk, and the exact search (every bracket missed, the
particles having moved together or apart between two passes).

Bars as in the parity tests: neighbour sets, distances and h bit-exact, density
and sound speed 1e-12 (plain FP64) and 1e-5 (FP32C) relative, bitwise form
exact.  The reference divides by that distance in the force, so accelerations of
the particles at one point are NaN there and in the FP64 forms, theirs alone;
FP32C keeps every acceleration finite.
"""
import numpy as np
import pytest

import oracle as O
from sphugo_amd import _lib as L
from sphugo_amd import ics

from test_gpu_parity import _check_knn, _rel

pytestmark = pytest.mark.gpu

FORMS = {"fp64": dict(precision=L.PREC_FP64), "fp32c": dict(precision=L.PREC_FP32C),
         "bitwise": dict(flags=L.FLAG_BITWISE)}


def _state(n, seed, at):
    """Uniform, with `at` consecutive particles at one point from every tenth
    of the array on."""
    st = ics.uniform(n, seed=seed)
    g = np.random.default_rng(seed)
    st["vx"], st["vy"] = 0.1 * g.standard_normal(n), 0.1 * g.standard_normal(n)
    same = np.zeros(n, bool)
    for i in range(0, n - at, n // 10):
        for f in ("x", "y"):
            st[f][i:i + at] = st[f][i]
        same[i:i + at] = True
    return st, same


def _check(g, o, same, form):
    _check_knn(g, o)
    bar = {"fp64": 1e-12, "fp32c": 1e-5, "bitwise": 0.0}[form]
    for f in ("rho", "c"):
        assert np.isfinite(o.get(f)).all()
        assert _rel(g.get(f), o.get(f)).max() <= bar, f
    for f in ("ax", "ay", "edot"):
        a, b = g.get(f), o.get(f)
        assert np.isfinite(b[~same]).all()
        assert np.isfinite(a if form == "fp32c" else a[~same]).all(), f
        assert np.abs(a - b)[~same].max() <= bar * np.abs(b[~same]).max(), f


@pytest.mark.parametrize("move", [1.0, 1.25, 1 / 1.2])
@pytest.mark.parametrize("n,k,at,kernel", [(257, 5, 2, 0), (2203, 32, 2, 1), (4099, 64, 3, 0),
                                           (30011, 19, 2, 1)])
@pytest.mark.parametrize("form", list(FORMS))
def test_density_beside_a_coincident_particle(form, n, k, at, kernel, move):
    st, same = _state(n, n + k, at)
    phys = dict(k=k, kernel=kernel, mass=st["mass"], gamma=5 / 3, visc_alpha=1.0, visc_beta=2.0,
                dt_half=0.001, hor=(-L.DBL_MAX, L.DBL_MAX), vert=(-L.DBL_MAX, L.DBL_MAX))
    init = [st[f] for f in ("x", "y", "vx", "vy", "e")]
    g = L.Sim(L.default_params(**phys, **FORMS[form]), *init)
    o = O.OracleSim(O.default_params(knn_mode=O.KNN_EXACT, **phys), *init)
    for s in (g, o):
        for f, v in (("vpx", st["vx"]), ("vpy", st["vy"]), ("epred", st["e"])):
            s.set(f, v)
        s.calculate_forces()  # the first pass
    _check(g, o, same, form)
    for f in ("x", "y"):
        for s in (g, o):
            s.set(f, st[f] * move)
    c0 = g.knn_counters()
    g.calculate_forces()
    c1 = g.knn_counters()
    o.calculate_forces()
    if move != 1.0:  # no h is within its bracket
        assert c1["retries"] - c0["retries"] >= n
    _check(g, o, same, form)


def test_fp32c_steps_over_coincident_particles():
    """At rest a pair stays together: steps of FP32C go on past it, in the walk
    and where one of the two misses its bracket."""
    st, _ = _state(2203, 5, 2)
    p = L.default_params(k=32, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                         vert=(0, 1), visc_alpha=1.0, visc_beta=2.0, precision=L.PREC_FP32C)
    g = L.Sim(p, st["x"], st["y"], np.zeros(2203), np.zeros(2203), st["e"])
    g.step(30)
    for f in ("x", "y", "vx", "vy", "e", "rho", "h", "ax", "ay", "edot"):
        assert np.isfinite(g.get(f)).all(), f
