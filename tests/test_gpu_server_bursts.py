"""Several passes between two admissions of the serve loop (GPU): jobs that arrive or
fail in the middle of such a run of passes leave every result what it is alone, and
where a pass is long an arrival waits for one pass at most."""
import time

import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def _p(n, **kw):
    kw.setdefault("dt_half", 0.0)
    return L.default_params(**{**dict(k=16, mass=1.0 / n, gamma=5 / 3, cfl=0.3, hor=(0, 1),
                                      vert=(0, 1), visc_alpha=1.0, visc_beta=2.0), **kw})


def _alone(p, st, nsteps):
    a = L.Sim(p, st["x"], st["y"], st["vx"], st["vy"], st["e"])
    a.step(nsteps)
    return {f: a.get(f) for f in L.RESULT_FIELDS}, a.reductions()


def _check(srv, j, p, st, nsteps):
    srv.wait(j, timeout=60)
    ref, red = _alone(p, st, nsteps)
    for f in L.RESULT_FIELDS:
        assert (srv.result(j, f) == ref[f]).all(), f
    assert (srv.reductions(j)[:6] == red).all()


def test_jobs_that_arrive_while_another_runs():
    srv = L.Server(20000, max_jobs=8, kmax=16)
    jobs = []
    for i, (n, nsteps) in enumerate([(3001, 1501), (1000, 7), (257, 1), (2048, 10), (1500, 2),
                                     (900, 33)]):
        st = ics.blast(n, seed=50 + i)
        p = _p(n, dt_half=1e-5)
        jobs.append((srv.submit(p, st, nsteps), p, st, nsteps))
        time.sleep(0.0023)
    assert srv.info(jobs[0][0])["state"] == "running"
    for j in jobs:
        _check(srv, *j)


def test_failure_between_two_looks_at_the_flags():
    """A particle that crosses three boxes per step is wrapped by one: it leaves the
    images in step 2, the second of the passes that follow the admission at once.  Its
    job fails, and those beside it do not notice."""
    bad = ics.uniform(2000, seed=9)
    bad["x"][17], bad["vx"] = 0.1, np.zeros(2000)
    bad["vx"][17] = 1500.0
    bad["e"] = np.full(2000, 1e-6)
    pbad = _p(2000, dt_half=1e-3, visc_alpha=0.0, visc_beta=0.0)
    a = L.Sim(pbad, bad["x"], bad["y"], bad["vx"], None, bad["e"])
    a.step(1)
    with pytest.raises(L.SphError, match="left the periodic images"):
        a.step(1)
    bad["vy"] = None
    srv = L.Server(20000, max_jobs=8, kmax=16)
    good = []
    for i, n in enumerate((2500, 1000, 4000)):
        st = ics.blast(n, seed=70 + i)
        good.append((srv.submit(_p(n), st, 25 + i), _p(n), st, 25 + i))
    jbad = srv.submit(pbad, bad, 40)
    with pytest.raises(L.SphError, match="left the periodic images"):
        srv.wait(jbad, timeout=60)
    for j in good:
        _check(srv, *j)
    s = srv.stats()
    assert s["jobs_done"] == 3 and s["jobs_failed"] == 1
    # its range and slot serve the next job
    st = ics.blast(2000, seed=80)
    _check(srv, srv.submit(_p(2000), st, 3), _p(2000), st, 3)


def test_arrivals_wait_for_one_pass_of_a_large_job():
    """Beside two million particles a job that arrives is admitted after the pass that
    runs, half a pass away on average."""
    n, nsteps = 2000000, 300
    st, small = ics.uniform(n, seed=1), ics.uniform(300, seed=2)
    srv = L.Server(n + 4096, max_jobs=8, kmax=16)
    big = srv.submit(_p(n, dt_half=1e-9), st, nsteps)
    while srv.info(big)["steps"] < 2:
        time.sleep(0.002)
    r = np.random.default_rng(0)
    waits = []
    for _ in range(20):
        j = srv.submit(_p(300, dt_half=1e-9), small, 1)
        srv.wait(j, timeout=60)
        waits.append(srv.info(j)["queue_ms"])
        time.sleep(float(r.uniform(0.004, 0.008)))
    assert srv.info(big)["state"] == "running"
    srv.wait(big, timeout=60)
    one = srv.info(big)["run_ms"] / (nsteps + 1)
    assert np.median(waits) < 1.2 * one, (one, waits)
