"""GPU: transfers to and from ordinary host memory. Values must not depend on how the bytes travel: through
the kernel's own page-locked reads and writes (small calls), one block, several, blocks used more than
once, or the runtime (more transfers at a time than there are blocks)."""
import threading

import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frame():
    return synth.random_cloud(20000, r=0.01, extent=0.3)


def points(xyz, r, n, seed):
    s = synth.Stream(seed)
    pick = (s.uniform(n) * len(xyz)).astype(np.int64)
    return (xyz[pick] + s.uniform(3 * n, -3 * r, 3 * r).reshape(-1, 3)).astype(np.float32)


# 44 n + 64 bytes: 256 KB is passed from 5957 points; 24 n bytes: a second block of 1 MB from 43691, a third (a group
# of one) from 87382, a ninth piece from 349526, an eleventh (a group of two and one of one) from 436907
@pytest.mark.parametrize("n", [1, 5956, 5957, 43690, 43691, 87382, 349525, 349526, 436907, 1000003])
def test_point_values_do_not_depend_on_the_transfer(frame, n):
    xyz, r = frame
    q = points(xyz, r, n, 5)
    ctx = gpu_context(xyz, r, precision=capi.FP32_KAHAN)
    f, g = ctx.eval_points(q, grad=True)
    f2 = ctx.eval_points(q)
    assert np.array_equal(f, f2)
    for a in sorted({0, max(0, n - 5000), max(0, n // 2 - 2500), max(0, min(n, (1 << 20) // 24) - 2500)}):
        fs, gs = ctx.eval_points(q[a:a + 5000], grad=True)
        assert np.array_equal(f[a:a + 5000], fs) and np.array_equal(g[a:a + 5000], gs), a
    ctx.close()


def test_threads_share_the_blocks(frame):
    """Four contexts in four threads ask for 32 blocks of 16."""
    xyz, r = frame
    q = [points(xyz, r, 200001, 20 + i) for i in range(4)]
    ctxs = [gpu_context(xyz, r) for _ in q]
    want = [ctxs[0].eval_points(x, grad=True) for x in q]
    got = [[] for _ in q]

    def work(i):
        for _ in range(5):
            got[i].append(ctxs[i].eval_points(q[i], grad=True))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for w, gs in zip(want, got):
        assert len(gs) == 5
        for g in gs:
            assert np.array_equal(w[0], g[0]) and np.array_equal(w[1], g[1])
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("n", [1, 4096, 4097, 300001])
def test_edges_by_pieces(frame, n):
    xyz, r = frame
    ctx = gpu_context(xyz, r)
    a = points(xyz, r, n, 31)
    b = a + np.float32(r) * np.eye(3, dtype=np.float32)[np.arange(n) % 3]
    ends = np.stack([np.concatenate([p, ctx.eval_points(p)[:, None]], axis=1) for p in (a, b)], axis=1)
    out, nev = ctx.bisect_edges(ends)
    for s in (slice(0, 2000), slice(max(0, n - 2000), n)):
        o, e = ctx.bisect_edges(ends[s])
        assert np.array_equal(out[s], o) and np.array_equal(nev[s], e)
    for at, bad in ((0, np.inf), (n // 2, np.nan), (n - 1, -np.inf)):
        e = ends.copy()
        e[at, 1, 3] = bad
        with pytest.raises(capi.PisurfError):
            ctx.bisect_edges(e)
    ctx.close()
