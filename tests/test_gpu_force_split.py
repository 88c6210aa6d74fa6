"""The force's two splits of the work (GPU): a thread per particle, or four
waves per 64 particles in small launches.

Both add a row's terms in the same four sections, so a small simulation gives
the same bits alone (four waves) and batched beside a large one (a thread per
particle), in every field and in the reductions.
"""
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def _p(st, k, prec, kernel):
    return L.default_params(k=k, mass=st["mass"], gamma=5 / 3, dt_half=0.0, cfl=0.3, hor=(0, 1),
                            vert=(0, 1), visc_alpha=1.0, visc_beta=2.0, precision=prec,
                            kernel=kernel)


# k: fewer chunks than sections, partial last chunks, uneven and even sections
@pytest.mark.parametrize("k", [4, 5, 12, 13, 19, 32, 63, 64])
@pytest.mark.parametrize("prec", [L.PREC_FP64, L.PREC_FP32C])
def test_split_equals_thread_per_particle(k, prec):
    sizes = [300, 449, 2200, 60000]  # last items of 44, 193 and 152 particles
    sts = [ics.blast(n, seed=n + k) for n in sizes]
    ps = [_p(st, k, prec, i % 2) for i, st in enumerate(sts)]
    b = L.Batch(ps, sts)
    b.step(2)
    for i, (p, st) in enumerate(zip(ps[:-1], sts)):
        a = L.Sim(p, st["x"], st["y"], st["vx"], st["vy"], st["e"])
        a.step(2)
        for f in L.FIELDS:
            assert (b.get_sim(i, f) == a.get(f)).all(), (i, f)
        assert (b.reductions_sim(i) == a.reductions()).all(), i


# the last size of one split and the first of the other, at k = 32
@pytest.mark.parametrize("n", [128 * 256, 128 * 256 + 1])
def test_batched_equals_alone_at_the_limit(n):
    sts = [ics.uniform(300, seed=n), ics.blast(n, seed=n + 1)]
    ps = [_p(st, 32, L.PREC_FP64, 0) for st in sts]
    b = L.Batch(ps, sts)
    b.step(2)
    a = L.Sim(ps[1], sts[1]["x"], sts[1]["y"], sts[1]["vx"], sts[1]["vy"], sts[1]["e"])
    a.step(2)
    for f in L.FIELDS:
        assert (b.get_sim(1, f) == a.get(f)).all(), f
