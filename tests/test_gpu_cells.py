"""Cell ranges and keys at the edges of their launches (GPU).

The cell ranges are written by blocks of their own, each for the cells of one
or more work items of a simulation; a single simulation's keys are made by the
sort's first launch in a range of sizes.  Neither may change a bit: a
simulation equals itself within a batch, where its items share a block with
other simulations' and its keys come from their own launch.
"""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

from test_gpu_edge import _pair
from test_gpu_parity import _check_knn

pytestmark = pytest.mark.gpu


def _p(st, k):
    return L.default_params(k=k, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                            vert=(0, 1), visc_alpha=1.0, visc_beta=2.0)


def _same(b, i, first, p, st, steps):
    a = L.Sim(p, st["x"], st["y"], st["vx"], st["vy"], st["e"])
    a.step(steps)
    for f in L.FIELDS:
        assert (b.get_sim(i, f) == a.get(f)).all(), (i, f)
    ids, _ = b.neighbours(with_d2=False)
    ia, _ = a.neighbours(with_d2=False)
    assert (ids[first:first + len(st["x"]), :p.k] == ia).all(), i


@pytest.mark.parametrize("n", [8192, 8193, 524288, 524289])
def test_alone_equals_batched_where_the_keys_move(n):
    sts = [ics.uniform(300, seed=n), ics.blast(n, seed=n + 1)]
    ps = [_p(s, 16) for s in sts]
    b = L.Batch(ps, sts)
    b.step(2)
    _same(b, 1, 300, ps[1], sts[1], 2)


def test_many_small_simulations_share_blocks():
    """2,200 simulations: two work items per block of cell ranges, with one
    simulation of several items among them."""
    sizes = [17 + i % 9 for i in range(2199)]
    sizes.insert(1100, 3000)
    sts = [ics.uniform(n, seed=i) for i, n in enumerate(sizes)]
    ps = [_p(s, 8) for s in sts]
    b = L.Batch(ps, sts)
    b.step(2)
    offs = np.concatenate([[0], np.cumsum(sizes)])
    for i in (0, 1, 1099, 1100, 1101, 2198, 2199):
        _same(b, i, int(offs[i]), ps[i], sts[i], 2)


@pytest.mark.parametrize("n,spread", [(5000, 1e-6), (30000, 1e-4)])
def test_one_crowded_cell(n, spread):
    """Nearly every particle in one cell, the other cells empty: the ranges of
    almost all cells come from blocks with no particle of their own."""
    rng = np.random.default_rng(n)
    st = dict(x=0.3 + spread * rng.random(n), y=0.7 + spread * rng.random(n), vx=np.zeros(n),
              vy=np.zeros(n), e=np.full(n, 10.0), mass=1.0 / n)
    st["x"][-3:], st["y"][-3:] = (0.999, 0.5, 0.02), (0.001, 0.02, 0.97)
    g, o = _pair(st, 8)
    _check_knn(g, o)
