"""The radix sort's forms at their size limits (GPU): one block, two launches
per pass with 2, 4 or 8 keys per thread, three launches per pass.

The sort is stable, so a simulation's particles come out in the same order
whichever form runs: a simulation batched with another so that their total
lies at a limit equals its standalone run bit for bit, in every field and in
its neighbour rows.
"""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def _p(st, k):
    return L.default_params(k=k, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                            vert=(0, 1), visc_alpha=1.0, visc_beta=2.0)


@pytest.mark.parametrize("total", [4097, 8191, 8192, 8193, 262144, 262145, 524288, 524289, 1048576,
                                   1048577])
def test_batched_equals_alone_at_sort_limits(total):
    sts = [ics.blast(2200, seed=total), ics.uniform(total - 2200, seed=total + 1)]
    ps = [_p(sts[0], 32), _p(sts[1], 16)]
    b = L.Batch(ps, sts)
    b.step(2)
    ids, _ = b.neighbours(with_d2=False)
    first = 0
    for i, (p, st) in enumerate(zip(ps, sts)):
        a = L.Sim(p, st["x"], st["y"], st["vx"], st["vy"], st["e"])
        a.step(2)
        for f in L.FIELDS:
            assert (b.get_sim(i, f) == a.get(f)).all(), (i, f)
        ia, _ = a.neighbours(with_d2=False)
        rows = ids[first:first + len(st["x"]), :p.k]
        assert (rows == ia).all(), i
        # the rows name every particle of the simulation's own range
        assert np.unique(ia).max() < len(st["x"])
        first += len(st["x"])
