"""What readbacks hold and use besides their bytes (GPU): pinned host memory and
host threads."""
import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu


def _sim(n, k=2, **kw):
    st = ics.uniform(n, seed=n)
    return L.Sim(L.default_params(k=k, mass=1.0 / n, hor=(0, 1), vert=(0, 1), **kw), st["x"],
                 st["y"], e=st["e"])


def _vm_size():
    with open("/proc/self/status") as f:
        return next(int(v.split()[1]) << 10 for v in f if v.startswith("VmSize:"))


def test_open_handles_hold_no_staging():
    """A call's pinned blocks are free for the next handle's when it ends: 24
    handles, open together, that each read more than a small copy's 256 KiB map
    less than 2 MiB each (a ring of slots has 8)."""
    sims = [_sim(40000) for _ in range(25)]
    sims[0].get("x")
    before = _vm_size()
    for g in sims[1:]:
        g.get("x")
    assert _vm_size() - before < 24 * (2 << 20)
