"""First passes (GPU): queries without an h get one from the candidates staged
for their group, within a radius guessed from the grid, before the walk.

The cases are the guess's bad ones: density contrasts far beyond a cell's
count, lists that hold nearly every particle, support radii of more than a
box, lattices full of ties, and lone particles between crowds.  The
neighbour sets, squared distances and h equal the oracle's whatever the guess
was, and a batched simulation equals itself alone bit for bit.
"""
import numpy as np
import pytest

from sphugo_amd import _lib as L

from test_gpu_edge import _lattice, _pair
from test_gpu_parity import _check_knn

pytestmark = pytest.mark.gpu


def _state(x, y):
    n = len(x)
    z = np.zeros(n)
    return dict(x=x, y=y, vx=z, vy=z.copy(), e=np.full(n, 10.0), mass=1.0 / n)


def _contrast(n, seed):
    """Log-uniform distances from three centres, and a few lone particles."""
    rng = np.random.default_rng(seed)
    c = rng.random((3, 2))[rng.integers(0, 3, n)]
    r = 10.0 ** rng.uniform(-6, -0.5, n)
    a = rng.uniform(0, 2 * np.pi, n)
    x, y = (c[:, 0] + r * np.cos(a)) % 1.0, (c[:, 1] + r * np.sin(a)) % 1.0
    x[:5], y[:5] = rng.random(5), rng.random(5)
    return _state(x, y)


def _uniform(n, seed):
    rng = np.random.default_rng(seed)
    return _state(rng.random(n), rng.random(n))


CASES = {
    "all-but-one": (lambda: _uniform(33, 1), 32, {}),
    "wider-than-the-box": (lambda: _uniform(9, 2), 32, {}),
    "thin-box": (lambda: _uniform(500, 3), 64, dict(hor=(0, 40))),
    "contrast-k2": (lambda: _contrast(3000, 4), 2, {}),
    "contrast-k64": (lambda: _contrast(20000, 5), 64, {}),
    "lattice": (lambda: _lattice(48), 32, {}),
}


@pytest.mark.parametrize("flags", [0, L.FLAG_BITWISE])
@pytest.mark.parametrize("case", CASES)
def test_first_pass_neighbours_are_exact(case, flags):
    make, k, kw = CASES[case]
    g, o = _pair(make(), k, flags=flags, **kw)
    _check_knn(g, o)


def test_first_pass_batched_equals_alone():
    cases = [c for c in CASES.values() if not c[2]]
    sts = [make() for make, _, _ in cases]
    ps = [L.default_params(k=k, mass=st["mass"], hor=(0, 1), vert=(0, 1)) for st, (_, k, _) in
          zip(sts, cases)]
    b = L.Batch(ps, sts)
    b.calculate_forces()
    for i, (p, st) in enumerate(zip(ps, sts)):
        a = L.Sim(p, st["x"], st["y"], st["vx"], st["vy"], st["e"])
        a.calculate_forces()
        for f in L.FIELDS:
            assert (b.get_sim(i, f) == a.get(f)).all(), (i, f)
