"""GPU: the particle normals that trees of 2^20 particles and more read. Before each tree the context takes the normals of
as many particles strewn over the same box: a normal that the tree reads without taking it has some other direction."""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


def stale_context(xyz, r, **kw):
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    u = synth.Stream(77).uniform(xyz.size).reshape(xyz.shape)
    ctx = gpu_context((lo + u * (hi - lo)).astype(np.float32), r, **kw)
    ctx.particle_normals()
    ctx.upload(xyz)
    ctx.reset_stats()
    return ctx


def tree(ctx):
    info = ctx.build_tree()
    return info, ctx.tree_nodes(info["n_nodes"])


def assert_same(a, b):
    assert a[0]["n_nodes"] == b[0]["n_nodes"]
    for key in ("type", "id", "depth", "child", "node"):
        assert np.array_equal(a[1][key], b[1][key]), key


@pytest.mark.parametrize("depth", [1, 2, 3])
def test_shallow_tree_takes_its_normals(depth):
    """A tree of depth 1 or 2 has all its levels below D_min, one of depth 3 has D_min at its root. A flat surface
    through the root box, which holds one layer of particles with equal normals: the root is a leaf."""
    r = 0.005
    i, j, k = np.meshgrid(np.arange(128), np.arange(128), np.arange(65), indexing="ij")
    p = np.stack([i, j, k - 64], axis=-1).reshape(-1, 3) * (2 * r)
    # the top layer lies at z = 0 and the surface at 0.95 r; one particle above puts the box's centre a little
    # more than the root's half width 2^(depth - 1) r above the layer
    p = np.concatenate([p, [[127 * r, 127 * r, 128 * r + 2 * (2 ** (depth - 1) + 0.05) * r]]])
    assert len(p) >= 1 << 20
    out = []
    for before in (False, True):
        ctx = stale_context(p.astype(np.float32), r, depth_max_override=depth)
        if before:
            ctx.particle_normals()
        out.append(tree(ctx))
        ctx.close()
    assert out[0][0]["depth_max"] == depth and out[0][0]["depth_min"] == depth - 3
    assert_same(*out)
    assert out[0][0]["n_nodes"] == 1


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP32_KAHAN, capi.FP64])
def test_later_trees_keep_the_normals(prec):
    """Trees built again on the same particles, each reading cells that the ones before did not, then a sweep that reads
    any: every tree as with all normals there before, every particle's normal counted once."""
    xyz, r = synth.crown_splash(pool_layers=6, n_drops=20000)
    assert len(xyz) >= 1 << 20
    kinds = [dict(smooth_factor=0.5), dict(qef_mode=capi.QEF_REFERENCE), dict(smooth_factor=3.0), dict()]
    out = []
    for before in (False, True):
        ctx = stale_context(xyz, r, precision=prec)
        if before:
            ctx.particle_normals()
        trees = []
        for kw in kinds:
            ctx.set_params(r, precision=prec, **kw)
            trees.append(tree(ctx))
            assert ctx.stats()["grad_evals"] == len(xyz)
        nodes = trees[-1][1]
        pick = np.arange(0, len(nodes["half"]), 97)
        level = ctx.sweep_level(nodes["center"][pick], nodes["half"][pick], np.full(len(pick), 20))
        assert ctx.stats()["grad_evals"] == len(xyz)
        out.append((trees, level))
        ctx.close()
    (ta, la), (tb, lb) = out
    for a, b in zip(ta, tb):
        assert_same(a, b)
    for a, b in zip(la, lb):
        assert np.array_equal(a, b)
    # the trees differ, so that later ones read more
    assert len({t[0]["n_nodes"] for t in ta}) > 1


def test_normals_left_out_between_trees():
    """A tree without normals in between clears them: the next tree takes its own again."""
    xyz, r = synth.crown_splash(pool_layers=6, n_drops=20000)
    ctx = stale_context(xyz, r)
    first = tree(ctx)
    ctx.set_params(r, calc_normals=False)
    flat = tree(ctx)
    ctx.set_params(r)
    assert_same(first, tree(ctx))
    assert flat[0]["n_nodes"] != first[0]["n_nodes"]
    ctx.close()


def test_a_tree_and_all_normals_tune_apart():
    """The shape kept for a tree's normals, timed on a launch with few runs at work, is not the one of all particles'."""
    xyz, r = synth.crown_splash(pool_layers=6, n_drops=20000)
    ctx = gpu_context(xyz, r)
    was = ctx.L.pisurf_run_tuning(1, 1)
    assert was == 0
    ctx.build_tree()
    kept = ctx.L.pisurf_run_tuning(-1, 0)
    ctx.particle_normals()
    assert ctx.L.pisurf_run_tuning(-1, 0) == kept + 1
    ctx.particle_normals()
    assert ctx.L.pisurf_run_tuning(-1, 0) == kept + 1
    ctx.close()
