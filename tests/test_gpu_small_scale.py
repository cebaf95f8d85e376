"""GPU: FP64 sums of frames so small that the square of a length is no normal float: what the sums by waves of points
leave out may not depend on it."""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -69, 2.0 ** -70])
def test_small_frames_by_waves_and_by_points(scale):
    """r = 0.01, 1.7e-23 and 8.5e-24 (half of that is too small for the anisotropy). 2^18 points or more go 64 to a wave,
    fewer a wave each. The scales are powers of two, so that the float positions are those of the first frame scaled."""
    xyz, r = synth.random_cloud(1500, r=0.01, extent=0.2)
    s = synth.Stream(41)
    n = (1 << 18) + 5
    q = (xyz[(s.uniform(n) * len(xyz)).astype(np.int64)] + s.uniform(3 * n, -3 * r, 3 * r).reshape(-1, 3)).astype(np.float32)
    f32 = np.float32
    xyz, q, r = xyz * f32(scale), q * f32(scale), float(f32(r) * f32(scale))
    ctx = gpu_context(xyz, r, precision=capi.FP64)
    whole = ctx.eval_points(q)
    assert np.all(np.isfinite(whole)) and np.count_nonzero(whole < 0.5 * whole.max()) > n // 10
    for a in range(0, n, 60000):
        assert np.array_equal(whole[a:a + 60000], ctx.eval_points(q[a:a + 60000])), a
    ctx.close()
