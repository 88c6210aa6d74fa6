"""Readback staging at its size limits (GPU): the one-block copy, the slots of
the ring (one to more than it holds, a last slot of any length), with one, two
and four host threads, and from several threads at once.  What was written is
read back bit for bit."""
import threading

import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def _sim(n, k=2):
    st = ics.uniform(n, seed=n)
    return L.Sim(L.default_params(k=k, mass=1.0, hor=(0, 1), vert=(0, 1)), st["x"], st["y"])


@pytest.mark.parametrize("n", [2, 3, 32767, 32768, 32769, 131072, 131073, 262143, 524289,
                               1048576, 1048577, 1179651, 2359301])
def test_fields_round_trip(n):
    g = _sim(n)
    r = np.random.default_rng(n)
    for f in ("vx", "e"):
        v = r.standard_normal(n)
        g.set(f, v)
        assert (g.get(f) == v).all(), f
    # into memory that was there already, and starts at an odd address
    raw = np.full(8 * n + 24, 7, np.uint8)
    for off in (8, 1):
        buf = np.frombuffer(raw.data, np.uint8)[off:off + 8 * n]
        L.check(L.lib().sph_read_field(g._h, L.FIELD["e"],
                                       buf.ctypes.data_as(L._D)))
        assert (np.frombuffer(buf.tobytes(), np.float64) == v).all()
        assert raw[off - 1] == 7 and (raw[off + 8 * n:] == 7).all()
        raw[:] = 7


def test_neighbour_rows_of_odd_length():
    g = _sim(10007, k=7)
    g.calculate_forces()
    ids, d2 = g.neighbours()
    only, _ = g.neighbours(with_d2=False)
    assert (ids == only).all() and (np.diff(d2, axis=1) >= 0).all()
    assert (d2[:, -1] ** 0.5 == g.get("h")).all()


def test_reads_from_several_threads():
    sims = [_sim(n) for n in (3000, 200001, 1500001)]
    vals = []
    for i, g in enumerate(sims):
        v = np.random.default_rng(i).standard_normal(g.n)
        g.set("vy", v)
        vals.append(v)
    bad = []

    def read(g, v):
        for _ in range(5):
            if not (g.get("vy") == v).all():
                bad.append(g.n)

    ts = [threading.Thread(target=read, args=a) for a in zip(sims, vals)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("ks", [(2,), (32,), (33,), (64,), (31, 64), (16, 32)])
def test_neighbour_rows_of_each_width(ks):
    """Rows of 32 and 64 lanes, alone and in batches of mixed k, on lattices
    (exact ties) and in boxes so small that a particle is its neighbours'
    neighbour through several images: ascending (d2, ID), the oracle's IDs and
    distances, positions at those distances, and the fill past a row's k."""
    import oracle as O
    sts, ps = [], []
    for i, k in enumerate(ks):
        a = (np.arange(13) + 0.5) / 13
        x, y = [v.ravel().copy() for v in np.meshgrid(a, a, indexing="ij")]
        if i % 2:
            x, y = ics.uniform(37, seed=k)["x"], ics.uniform(37, seed=k)["y"]
        n = len(x)
        sts.append({"x": x, "y": y, "vx": np.zeros(n), "vy": np.zeros(n), "e": np.ones(n)})
        ps.append(L.default_params(k=k, mass=1.0 / n, hor=(0, 1), vert=(0, 1)))
    g = L.Batch(ps, sts)
    g.calculate_forces()
    ids, d2 = g.neighbours()
    px, py = g.neighbour_pos()
    first = 0
    for k, st in zip(ks, sts):
        n = len(st["x"])
        o = O.OracleSim(O.default_params(knn_mode=O.KNN_EXACT, k=k, mass=1.0 / n, hor=(0, 1),
                                         vert=(0, 1)), st["x"], st["y"], st["vx"], st["vy"], st["e"])
        o.calculate_forces()
        oi, od = o.neighbours()
        rows = slice(first, first + n)
        assert (ids[rows, :k].astype(np.int64) == oi).all() and (d2[rows, :k] == od).all()
        q = (st["x"][:, None] - px[rows, :k]) ** 2 + (st["y"][:, None] - py[rows, :k]) ** 2
        assert np.abs(q - od).max() <= 1e-14
        assert (ids[rows, k:] == 0xFFFFFFFF).all() and np.isnan(d2[rows, k:]).all()
        assert np.isnan(px[rows, k:]).all() and np.isnan(py[rows, k:]).all()
        first += n


@pytest.mark.parametrize("n", [3, 8191, 8192, 8193])
def test_small_fields_in_order(n):
    """Either side of the most values ordered in LDS: alone and in a batch
    behind another simulation, with IDs in a shuffled input order, after steps
    that permute the particles."""
    r = np.random.default_rng(n)
    sts = [ics.uniform(m, seed=m) for m in (1001, n)]
    ps = [L.default_params(k=2, mass=1.0 / len(s["x"]), hor=(0, 1), vert=(0, 1))
          for s in sts]
    b = L.Batch(ps, sts)
    ids = r.permutation(n).astype(np.uint32)
    st, p = sts[1], ps[1]
    g = L.Sim(p, st["x"], st["y"], ids=ids)
    g.calculate_forces()
    b.calculate_forces()
    assert (b.get_sim(1, "x") == st["x"]).all() and (b.get_sim(0, "y") == sts[0]["y"]).all()
    assert (g.get("x")[ids] == st["x"]).all() and (g.get("y")[ids] == st["y"]).all()
    v = r.standard_normal(n)
    g.set("e", v)
    assert (g.get("e") == v).all()
