"""Neighbour readback of a state gone bad (GPU): a particle whose position is no
number has no distances, and its row still leaves whole: every entry written,
each of its neighbours once."""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(3000, 12), (3000, 33), (301, 64)])
def test_row_of_a_particle_without_a_position(n, k):
    st = ics.uniform(n, seed=n + k)
    g = L.Sim(L.default_params(k=k, mass=1.0 / n, hor=(0, 1), vert=(0, 1)), st["x"], st["y"],
              e=st["e"])
    g.calculate_forces()
    g.neighbours()
    g.neighbour_pos()
    bad = n // 3
    vx = np.zeros(n)
    vx[bad] = np.nan
    g.set("vx", vx)
    with pytest.raises(L.SphError, match="left the periodic images"):
        g.step(1)
    ids, d2 = g.neighbours()
    px, py = g.neighbour_pos()
    assert np.isnan(d2[bad]).all() and np.isfinite(np.delete(d2, bad, 0)).all()
    assert (ids < n).all() and (np.diff(np.sort(ids, axis=1).astype(np.int64), axis=1) > 0).all()
    for v, w in ((px, "x"), (py, "y")):
        assert v.shape == ids.shape
        assert (np.isfinite(v[bad]) | (ids[bad] == bad)).all(), w
