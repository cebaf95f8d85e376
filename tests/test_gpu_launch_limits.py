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


@pytest.mark.parametrize("side", [16370, 16400])
def test_lattice_of_a_sheet(side):
    """Five points thick and 1.3 G points in all: 2^24 blocks of 16 x 4 x 4 points hold fewer or more than that."""
    r = 2.0 ** -8
    lo = np.array([0.5, 0.25, 0.25])
    ends = lo + r * np.array([[0.0, 0.0, 0.0], [0.0, side, side]])
    # (on the sheet, so that the box stays as thick as one particle's)
    flat = np.array([[0.0, a, b] for a in (0.0, 1.5, 3.0, side - 2.0) for b in (0.0, 2.0, side - 4.0)])
    xyz = np.concatenate([ends, lo + r * flat]).astype(np.float32)
    ctx = gpu_context(xyz, r)
    vals, box, sp = ctx.uniform_grid()
    nz, ny, nx = vals.shape
    blocks = -(-nx // 16) * -(-ny // 4) * -(-nz // 4)
    assert nx == 5 and (blocks >= 1 << 24) == (side > 16384)
    f32 = np.float32

    def axis(a, n, i):
        st = f32(n - 1)
        return (f32(n - 1 - i) / st) * f32(box[2 * a]) + (i.astype(f32) / st) * f32(box[2 * a + 1])

    away = np.ones((nz, ny), bool)
    seen = 0
    for y0 in (0, ny - 12):
        for z0 in (0, nz // 2, nz - 12):
            ys, zs = np.arange(y0, y0 + 12), np.arange(z0, z0 + 12)
            z, y, x = np.meshgrid(axis(2, nz, zs), axis(1, ny, ys), axis(0, nx, np.arange(nx)), indexing="ij")
            f = ctx.eval_points(np.stack([x, y, z], axis=-1).astype(f32).reshape(-1, 3)).astype(f32)
            part = vals[z0:z0 + 12, y0:y0 + 12]
            # (so few particles on a plane can have covariances of 0 / 0, whose records are NaN)
            assert np.array_equal(part.reshape(-1), f, equal_nan=True)
            seen += np.count_nonzero(part != vals[nz // 2, ny // 2, 2])
            away[z0:z0 + 12, y0:y0 + 12] = False
    ctx.close()
    assert seen > 0
    rows = np.flatnonzero(away.all(axis=1))
    assert np.all(vals[rows[0]:rows[-1] + 1:997] == vals[nz // 2, ny // 2, 2])
