"""An annulus too full to part (GPU): a query with more neighbours at exactly its
k-th distance than the walk's annulus holds goes to the exact search and weighs one
in the share of overflows that narrows the bracket."""
import numpy as np
import pytest

import oracle as O
from sphugo_amd import _lib as L

from test_gpu_parity import _check_knn

pytestmark = pytest.mark.gpu


def test_a_full_annulus_counts_once():
    # eight particles, each the centre of 36 at one distance: the points of integer
    # coordinates on a circle of 65, in steps of 2^-14 (differences are exact)
    ring = [(a, b) for a in range(-65, 66) for b in range(-65, 66) if a * a + b * b == 65 * 65]
    assert len(ring) == 36
    r = np.random.default_rng(3)
    x, y = [], []
    for i in range(8):
        for a, b in [(0, 0)] + ring:
            x.append((2 * i + 1) / 16 + a * 2.0 ** -14)
            y.append(3 / 32 + b * 2.0 ** -14)
    n = 1280
    m = n - len(x)
    x = np.concatenate([x, r.random(m)])
    y = np.concatenate([y, 0.3 + 0.6 * r.random(m)])
    st = [x, y, np.zeros(n), np.zeros(n), np.ones(n)]
    phys = dict(k=32, mass=1.0 / n, hor=(0, 1), vert=(0, 1))
    g = L.Sim(L.default_params(**phys), *st)
    o = O.OracleSim(O.default_params(knn_mode=O.KNN_EXACT, **phys), *st)
    o.calculate_forces()
    for _ in range(3):
        c0 = g.knn_counters()
        g.calculate_forces()
        c1 = g.knn_counters()
        _check_knn(g, o)
        assert c1["miss_ann"] - c0["miss_ann"] == 8
        # 8 of 1280 are less than 1/128 (10) and more than a quarter of it: the
        # bracket holds; twice as many would narrow it to 0.02
        assert L.get_tuning(g)["delta"] == 0.025
