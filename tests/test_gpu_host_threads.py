"""GPU: the threads that move large arrays to and from the caller's memory, and what they cost beside it."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

pytestmark = pytest.mark.gpu


def run(code):
    # a process of its own: the threads of the contexts of this one would be counted too
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout.split()


@pytest.mark.parametrize("cpus", [1, 2, 16])
def test_no_more_threads_than_processors(cpus):
    cpus = min(cpus, len(os.sched_getaffinity(0)))
    out = run("""
import os
import numpy as np
from particleisosurface_amd import capi, synth
xyz, r = synth.random_cloud(20000, r=0.01, extent=0.3)
ctx = capi.Context(0)
ctx.set_params(r)
ctx.upload(xyz)
q = np.tile(xyz, (60, 1))
ctx.eval_points(q[:100])
few = ctx.eval_points(q[:5000])  # the runtime's own threads are there
tasks = lambda: len(os.listdir("/proc/self/task"))
os.sched_setaffinity(0, sorted(os.sched_getaffinity(0))[:%d])
before = tasks()
f = ctx.eval_points(q)
print(tasks() - before)
assert np.array_equal(f[:5000], few) and np.array_equal(f[-20000:][:5000], few)
ctx.close()
""" % cpus)
    assert 0 <= int(out[0]) <= min(cpus, 8) - 1


def test_workers_sleep_while_a_kernel_runs():
    """The values of a lattice whose kernel takes far longer than their copy: the processor time of the call is the calling
    thread's, and what the copy takes, not eight threads' over the whole kernel."""
    out = run("""
import time
import numpy as np
from particleisosurface_amd import capi, synth
rng = np.random.default_rng(5)
r = 0.01
xyz = rng.uniform(0, 1.0, (400000, 3)).astype(np.float32)  # 25 particles a cell of 4 r
xyz = np.concatenate([xyz] * 8) + rng.uniform(0, 0.2 * r, (8 * len(xyz), 3)).astype(np.float32)
ctx = capi.Context(0)
ctx.set_params(r, precision=capi.FP64)
ctx.upload(xyz)
ctx.anisotropy()
ctx.uniform_grid()
ctx.uniform_grid()
best = []
for _ in range(5):
    t, c = time.perf_counter(), time.process_time()
    ctx.uniform_grid()
    best.append((time.perf_counter() - t, time.process_time() - c))
ctx.close()
t, c = min(best, key=lambda x: x[1] / x[0])
print(t, c)
""")
    t, c = float(out[0]), float(out[1])
    print("%.1f ms, %.1f ms of processors" % (1e3 * t, 1e3 * c))
    assert c < 2.5 * t
