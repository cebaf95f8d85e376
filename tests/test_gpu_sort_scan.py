"""GPU: the radix sort's and the scan's launch forms, at the sizes where they change."""
import numpy as np
import pytest

from particleisosurface_amd import synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


# tiles of 4096 keys: one, two, the most whose counts a tile adds up itself and one more, and more than
# 2048 (a complete scan)
@pytest.mark.parametrize("n", [4096, 4097, 262144, 262145, 8388609])
def test_sorted_particles(n):
    s = synth.Stream(n)
    xyz = s.uniform(3 * n, 0.0, 0.2).reshape(-1, 3).astype(np.float32)
    xyz[: n // 3] = xyz[n // 2]  # a digit that holds a third of the keys
    ctx = gpu_context(xyz, 0.001)
    g = ctx.hashgrid_build()
    il, _, _ = ctx.hashgrid_download(g["cellnum"])
    ctx.close()
    assert g["n_invalid"] == 0
    c = ((xyz - g["bounding"][0::2]) / np.float32(g["cellsize"])).astype(np.int64)
    key = (c[:, 2] * int(g["cellnum3"][1]) + c[:, 1]) * int(g["cellnum3"][0]) + c[:, 0]
    assert np.array_equal(il, np.argsort(key, kind="stable"))


# counts + 1 elements: one tile of 2048, one workgroup up to 16384, two launches above
@pytest.mark.parametrize("nq", [2047, 2048, 16383, 16384])
def test_list_offsets(nq):
    xyz, r = synth.random_cloud(3000, r=0.01, extent=0.15)
    s = synth.Stream(nq)
    q = s.uniform(3 * nq, 0.0, 0.15).reshape(-1, 3).astype(np.float32)
    ctx = gpu_context(xyz, r)
    ctx.hashgrid_build()
    off, ids = ctx.neighbors(q)
    parts = [ctx.neighbors(q[a:a + 1000]) for a in range(0, nq, 1000)]
    ctx.close()
    assert np.array_equal(np.diff(off), np.concatenate([np.diff(o) for o, _ in parts])) and off[0] == 0
    assert np.array_equal(ids, np.concatenate([i for _, i in parts]))
