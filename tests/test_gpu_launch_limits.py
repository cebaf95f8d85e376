"""GPU: calls whose threads, counted one kernel launch to a call, pass what a launch holds (2^32)."""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


def test_points_of_many_launches():
    """2^30 points and more are not sorted and take eight threads each (sixteen with FP64 gradients)."""
    n = (1 << 30) + 5
    xyz, r = synth.random_cloud(3000, r=0.01, extent=0.15)
    near = (xyz[:1500] + np.float32(0.3 * r)).astype(np.float32)
    q = np.full((n, 3), 9.0, np.float32)
    at = [0] + [(k << 27) - 700 for k in (1, 2, 5, 8)] + [n - len(near)]
    at[4] = n - 2 * len(near)  # (the last slice's few points end the last piece)
    for a in at:
        q[a:a + len(near)] = near
    ctx = gpu_context(xyz, r)
    want = ctx.eval_points(near)
    empty = ctx.eval_points(np.full((1, 3), 9.0, np.float32))[0]
    f = ctx.eval_points(q)
    ctx.close()
    for a in at:
        assert np.array_equal(f[a:a + len(near)], want), a
        f[a:a + len(near)] = empty
    assert np.all(f == empty)
