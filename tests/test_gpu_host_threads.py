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
