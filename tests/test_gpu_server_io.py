"""Admission and completion of served jobs (GPU), an upload and a launch each:
jobs whose last work item is full, holds one particle or is the only one, with
results on either side of the small readback, in reused slots and ranges,
equal their standalone runs bit for bit; velocities and energies left out read
as zero."""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def test_jobs_equal_standalone_runs_in_reused_slots():
    # 4,680 and 4,682 particles: 7 rows on either side of 256 KB
    sizes = [70001, 40, 256, 257, 4680, 4682, 512, 513, 40]
    srv = L.Server(72000, max_jobs=3, kmax=32)
    runs, ids = [], []
    for i, n in enumerate(sizes):
        st = ics.blast(n, seed=100 + i) if n > 1000 else ics.uniform(n, seed=100 + i)
        if i % 2:
            st["vx"] = st["vy"] = None
        p = L.default_params(k=16, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                             vert=(0, 1), visc_alpha=1.0, visc_beta=2.0)
        runs.append((p, st, 2 + i % 3))
        ids.append(srv.submit(p, st, runs[-1][2]))
    for j, (p, st, steps) in zip(ids, runs):
        srv.wait(j)
        n = len(st["x"])
        v = [np.zeros(n) if st[f] is None else st[f] for f in ("vx", "vy")]
        a = L.Sim(p, st["x"], st["y"], *v, st["e"])
        a.step(steps)
        for f in ("x", "y", "vx", "vy", "rho", "e", "h"):
            assert (srv.result(j, f) == a.get(f)).all(), (n, f)
        assert (srv.reductions(j)[:6] == a.reductions()).all()
        srv.release(j)
