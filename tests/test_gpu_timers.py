"""Kernel timers (GPU): a class that launches something counts once per pass, one
that launches nothing (the totals of a small launch, which its force makes, the keys
that one simulation's sort makes, the walk's former second launch) counts nothing
and takes no time."""
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,none", [(2200, {"reduce"}), (512 * 256, {"reduce", "keys"}),
                                    (512 * 256 + 1, {"keys"}), (2048 * 256 + 1, set())])
def test_timers_count_what_is_launched(n, none):
    st = ics.uniform(n, seed=4)
    p = L.default_params(k=16, mass=1.0 / n, hor=(0, 1), vert=(0, 1), flags=L.FLAG_TIMING)
    g = L.Sim(p, st["x"], st["y"], e=st["e"])
    g.step(2)  # three passes
    ms, count = g.kernel_times()
    for name in L.TIMERS:
        if name in none | {"knn_finish"}:
            assert ms[name] == 0 and count[name] == 0, name
        else:
            assert ms[name] > 0 and count[name] == 3, name
