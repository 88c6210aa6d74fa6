"""What readbacks hold and use besides their bytes (GPU): pinned host memory and
host threads."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from sphugo_amd import _lib as L
from sphugo_amd import ics

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


SHIM = r"""
#include <stddef.h>
int (*real)(void**, size_t, unsigned);
int calls;
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  ++calls;
  if (real) real(NULL, n, flags);  /* refused: leaves its error with the runtime */
  return 2;                        /* hipErrorOutOfMemory */
}
"""
CHILD = """
import ctypes, sys
import numpy as np
sys.path.insert(0, sys.argv[2])
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from sphugo_amd import _lib as L, ics
L.lib()
hip = next(v.split()[-1] for v in open("/proc/self/maps") if "libamdhip64" in v)
ctypes.c_void_p.in_dll(shim, "real").value = ctypes.cast(ctypes.CDLL(hip).hipHostMalloc,
                                                         ctypes.c_void_p).value


def params(n, k):
    return L.default_params(k=k, mass=1.0 / n, hor=(0, 1), vert=(0, 1))


for n in (3000, 8193, 40000, (1 << 20) + 1):
    st = ics.uniform(n, seed=n)
    g = L.Sim(params(n, 2), st["x"], st["y"], e=st["e"])
    assert (g.get("x") == st["x"]).all() and (g.get("y") == st["y"]).all()
    v = np.random.default_rng(n).standard_normal(n)
    g.set("e", v)
    assert (g.get("e") == v).all()
    g.close()
    print("field", n, flush=True)
st = ics.uniform(3001, seed=1)
g = L.Sim(params(3001, 7), st["x"], st["y"], e=st["e"])
g.step(3)
g.synchronize()
ids, d2 = g.neighbours()
px, py = g.neighbour_pos()
assert (np.diff(d2, axis=1) >= 0).all() and (d2[:, -1] ** 0.5 == g.get("h")).all()
assert px.shape == py.shape == ids.shape
c, red = g.knn_counters(), g.reductions()
assert c["failures"] == 0 and red[1] == red[1]
srv = L.Server(4000, max_jobs=2, kmax=8)
j = srv.submit(params(3001, 7), st, 3)
srv.wait(j, timeout=60)
for f in ("x", "y", "vx", "vy", "rho", "e", "h"):
    assert (srv.result(j, f) == g.get(f)).all(), f
assert (srv.reductions(j)[:6] == red).all()
srv.close()
assert ctypes.c_int.in_dll(shim, "calls").value > 0
print("whole", flush=True)
"""


def test_reads_without_pinned_memory(tmp_path):
    """Where no pinned memory is to be had, every read goes through the runtime's
    own copy: in a process of its own, whose hipHostMalloc refuses."""
    src, lib, prog = tmp_path / "shim.c", tmp_path / "libshim.so", tmp_path / "child.py"
    src.write_text(SHIM)
    prog.write_text(CHILD)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    r = subprocess.run([sys.executable, str(prog), str(lib), ROOT], capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1] == "whole", r.stdout + r.stderr[-2000:]


def test_waiting_for_the_gpu_takes_one_thread():
    """A large read behind a queue of steps: until they are done only the caller
    waits (its own wait is the runtime's, which may spin)."""
    g = _sim(1 << 20, k=16, dt_half=1e-9)
    g.step(1)
    g.get("x")
    g.step_async(300)
    wall, cpu = time.perf_counter(), time.process_time()
    g.get("x")
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.02  # long beside the copy itself
    assert cpu < 2 * wall
    g.synchronize()
