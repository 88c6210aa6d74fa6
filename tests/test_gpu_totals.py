"""Totals by the force's last block (GPU): small launches add a simulation's
totals up in the force's own launch, larger ones in launches of their own.

Held to sums of the fields read back, and bit for bit to the same simulation in a
launch of the other kind.  A total of positive terms goes through at most 30
roundings on either side (additions in trees over items and waves, the terms
themselves), so the sums agree to 64 * 2^-53.
"""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu

LIMIT = 512 * 256  # particles of the largest launch that finishes in the force
TOL = 64 * 2.0 ** -53


def _p(st, k=16):
    return L.default_params(k=k, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                            vert=(0, 1), visc_alpha=1.0, visc_beta=2.0)


def _sim(st):
    return L.Sim(_p(st), st["x"], st["y"], st["vx"], st["vy"], st["e"])


# one item, a whole one, one particle more, the limit and one particle past it
@pytest.mark.parametrize("n", [17, 256, 257, 2200, LIMIT, LIMIT + 1])
def test_totals_are_the_fields_sums(n):
    st = ics.blast(n, seed=n)
    s = _sim(st)
    for graph in (False, True, True):  # replayed with eager reads between
        L.set_graph(s, graph)
        s.step(2)
        f = {q: s.get(q) for q in ("vx", "vy", "e", "rho", "h", "c")}
        sp2 = f["vx"] ** 2 + f["vy"] ** 2
        red = s.reductions()
        want = [f["e"].sum(), f["rho"].sum(), (st["mass"] * (f["e"] + 0.5 * sp2)).sum()]
        for got, w in zip(red, want):
            assert abs(got - w) <= TOL * abs(w)
        # momenta cancel: held to the sum of their terms' sizes
        for got, v in zip(red[3:5], (f["vx"], f["vy"])):
            assert abs(got - st["mass"] * v.sum()) <= TOL * st["mass"] * np.abs(v).sum()
        cfl = (0.5 * f["h"] / (f["c"] + np.sqrt(sp2))).min()
        assert abs(s.next_dt_half() - 0.5 * 0.3 * cfl) <= 4 * 2.0 ** -53 * cfl


def test_small_and_large_launch_give_the_same_bits():
    sts = [ics.blast(n, seed=n) for n in (300, 2200, LIMIT)]
    b = L.Batch([_p(st) for st in sts], sts)  # past the limit together
    b.step(3)
    for i, st in enumerate(sts):
        a = _sim(st)
        a.step(3)
        assert (b.reductions_sim(i) == a.reductions()).all(), i
        for f in ("x", "vx", "rho"):
            assert (b.get_sim(i, f) == a.get(f)).all(), (i, f)
