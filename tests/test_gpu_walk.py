"""The bracketed kNN walk at the edges of its groups (GPU): item and group
remainders, few and many candidates per group (one to four rounds, boxes too
full for a group), the smallest and largest k, image-crossing groups, and
every wave width, against the oracle.

Each case finds h by the exact search, then walks the same state with the
bracket around it.  Bars on what the walk computes: neighbour sets, squared
distances and h bit-exact; density and sound speed 1e-12 (plain FP64) and 1e-5
(FP32C) relative.  Forces over the rows it writes are held in the parity tests.
"""
import numpy as np
import pytest

import oracle as O
from sphugo_amd import _lib as L
from sphugo_amd import ics

from test_gpu_parity import _check_knn, _pair, _rel

pytestmark = pytest.mark.gpu


def _clumps(n, seed):
    """Tight clumps on a sparse background: neighbouring queries of the curve
    lie far apart, and a group's box can hold whole clumps."""
    g = np.random.default_rng(seed)
    st = ics.uniform(n, seed=seed)
    m = 3 * n // 4
    c = g.random((5, 2))
    w = g.integers(0, 5, m)
    st["x"][:m] = (c[w, 0] + 2e-3 * g.standard_normal(m)) % 1.0
    st["y"][:m] = (c[w, 1] + 2e-3 * g.standard_normal(m)) % 1.0
    st["vx"], st["vy"] = 0.1 * g.standard_normal(n), 0.1 * g.standard_normal(n)
    return st


@pytest.mark.parametrize("n,k", [(17, 2), (33, 3), (241, 16), (255, 31), (257, 64), (272, 33),
                                 (4099, 2), (4099, 17), (4111, 64)])
@pytest.mark.parametrize("layout", ["uniform", "clumps"])
@pytest.mark.parametrize("prec", [L.PREC_FP64, L.PREC_FP32C])
def test_walk_edges(n, k, layout, prec):
    st = ics.uniform(n, seed=n + k) if layout == "uniform" else _clumps(n, n + k)
    g, o = _pair(st, k, precision=prec)
    h0 = g.get("h")
    seen = []
    for group in (64, 32, 16):
        # the bracket starts from the same width (it adapts after each pass)
        L.set_tuning(g, group=group, split=64 if k > 32 else 24, delta=0.025)
        g.calculate_forces()
        _check_knn(g, o)
        assert (g.get("h") == h0).all()
        bar = 1e-12 if prec == L.PREC_FP64 else 1e-5
        assert _rel(g.get("rho"), o.get("rho")).max() <= bar
        assert _rel(g.get("c"), o.get("c")).max() <= bar
        seen.append([g.get(f) for f in ("rho", "ax", "ay", "edot")])
    # the same bits however many groups a wave takes
    for a in seen[1:]:
        assert all((u == v).all() for u, v in zip(a, seen[0]))


def test_walk_resolves_most_queries():
    """At rest every bracket holds: what is left to the exact search is only
    what a group could not hold."""
    st = ics.clustered(30000, seed=3, k=64)
    g, _ = _pair(st, 64)
    c0 = g.knn_counters()
    g.calculate_forces()
    c1 = g.knn_counters()
    assert c1["retries"] - c0["retries"] <= st["n"] // 20, (c0, c1)


def _lattice(m):
    a = (np.arange(m) + 0.5) / m
    x, y = [v.ravel().copy() for v in np.meshgrid(a, a, indexing="ij")]
    n = m * m
    return {"x": x, "y": y, "vx": np.sin(40 * y), "vy": np.cos(30 * x), "e": 1.0 + x,
            "mass": 1.0 / n}


@pytest.mark.parametrize("name,k", [("lattice", 32), ("lattice", 40), ("lattice", 64),
                                    ("uniform", 2), ("uniform", 31), ("clumps", 64), ("tiny", 36),
                                    ("tiny", 64)])
def test_bitwise_walk_is_exact(name, k):
    """Bitwise form: the pass that walks gives the oracle's bits, as the pass of
    exact searches before it does, exact ties (lattice) and neighbours through
    several images (ten particles) included."""
    st = {"lattice": lambda: _lattice(24), "uniform": lambda: ics.uniform(4099, seed=k),
          "clumps": lambda: _clumps(4099, k), "tiny": lambda: ics.uniform(10, seed=4)}[name]()
    g, o = _pair(st, k, flags=L.FLAG_BITWISE)
    for _ in range(2):
        _check_knn(g, o)
        for f in ("rho", "c", "h", "ax", "ay", "edot"):
            assert (g.get(f) == o.get(f)).all(), f
        g.calculate_forces()


# open boxes whose particles move together or apart between two passes: the last
# h's bracket then holds k neighbours too many (squeezed beyond 1 + delta), too few
# (stretched), either from place to place, or more than its annulus takes (delta
# 0.1 at k = 64)
@pytest.mark.parametrize("move,delta", [(1 / 1.2, 0.025), (1 / 1.5, 0.1), (1.0, 0.1), (1.25, 0.025),
                                        ("mixed", 0.05)])
@pytest.mark.parametrize("layout,n,k", [("uniform", 257, 64), ("uniform", 4099, 33),
                                        ("lattice", 576, 40), ("clumps", 4111, 64)])
@pytest.mark.parametrize("prec", [L.PREC_FP64, L.PREC_FP32C])
def test_bracket_beside_the_kth_distance(move, delta, layout, n, k, prec):
    st = {"uniform": lambda: ics.uniform(n, seed=n + k), "lattice": lambda: _lattice(24),
          "clumps": lambda: _clumps(n, n + k)}[layout]()
    phys = dict(k=k, mass=st["mass"], gamma=5 / 3, visc_alpha=1.0, visc_beta=2.0, dt_half=0.001,
                hor=(-L.DBL_MAX, L.DBL_MAX), vert=(-L.DBL_MAX, L.DBL_MAX))
    init = [st[f] for f in ("x", "y", "vx", "vy", "e")]
    g = L.Sim(L.default_params(precision=prec, **phys), *init)
    o = O.OracleSim(O.default_params(knn_mode=O.KNN_EXACT, **phys), *init)
    for s in (g, o):
        for f, v in (("vpx", st["vx"]), ("vpy", st["vy"]), ("epred", st["e"])):
            s.set(f, v)
    g.calculate_forces()
    L.set_tuning(g, delta=delta)
    for f in ("x", "y"):
        v = st[f] * move if move != "mixed" else st[f] + 0.05 * np.sin(9 * st[f])
        g.set(f, v)
        o.set(f, v)
    c0 = g.knn_counters()
    g.calculate_forces()
    c1 = g.knn_counters()
    o.calculate_forces()
    _check_knn(g, o)
    bar = 1e-12 if prec == L.PREC_FP64 else 1e-5
    assert _rel(g.get("rho"), o.get("rho")).max() <= bar
    # an annulus too full needs no exact search
    if layout == "uniform" and move == 1:
        assert c1["retries"] - c0["retries"] <= n // 20, (c0, c1)
