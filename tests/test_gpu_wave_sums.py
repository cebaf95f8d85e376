"""GPU: sums by waves of 64 points (matrix-core cull) against one thread per point, bit for bit.

Levels of at least 2^18 sample points take the wave kernels; with sample_dedupe = 0 every sample is
summed by a thread of its own, in the same candidate order, so values, trees and meshes are equal.
The frame has a fluid surface, spray (waves over many rows, particles alone in their cells) and a
cluster whose windows hold more candidates than a wave stages at a time.
"""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def frame():
    xyz, r = synth.sloshing_tank(r=0.0045, n_spray=600)
    s = synth.Stream(91)
    blob = np.array([0.5, 0.25, 0.33]) + 3 * r * s.normal(3 * 3000).reshape(-1, 3)
    return np.concatenate([xyz, blob.astype(np.float32)]), r


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP32_KAHAN, capi.FP64])
@pytest.mark.parametrize("ani,poly6", [(True, False), (True, True), (False, True)])
def test_wave_sums_equal_per_point_sums(frame, prec, ani, poly6):
    xyz, r = frame
    out = []
    for dedupe in (True, False):
        ctx = gpu_context(xyz, r, precision=prec, use_ani=ani, use_poly6=poly6, sample_dedupe=dedupe)
        info = ctx.run_frame()
        out.append((info, ctx.tree_nodes(info["n_nodes"]), ctx.mesh(), ctx.stats()))
        ctx.close()
    (ia, na, ma, sa), (ib, nb, mb, sb) = out
    assert ia == ib
    # a level's distinct points pass the waves' lower bound
    assert sa["sample_unique"] > 2 * (1 << 18)
    for key in ("type", "id", "depth", "child", "node"):
        assert np.array_equal(na[key], nb[key]), key
    assert np.array_equal(ma[0], mb[0]) and np.array_equal(ma[1], mb[1])
    assert sa["field_evals"] == sb["field_evals"]


@pytest.mark.parametrize("nq", [1, 3, 4, 5, 257])
def test_neighbor_lists_of_few_queries(nq):
    """One wave per query: counts that leave waves of a workgroup without one, queries in a dense cluster
    (lists of several hundred ids), alone in their cells and off the grid, against the reference order."""
    xyz, r = synth.random_cloud(900, r=0.01, extent=0.1)
    far = np.array([[0.5, 0.5, 0.5], [0.5, 0.62, 0.5]], np.float32)
    xyz = np.concatenate([xyz, far])
    q = np.concatenate([far, xyz[:300], [[9.0, 0.0, 0.0]]]).astype(np.float32)[-nq:]
    ctx = gpu_context(xyz, r)
    ctx.hashgrid_build()
    off, ids = ctx.neighbors(q)
    from oracle.pyoracle import Oracle
    o = Oracle(xyz, r)
    o.hashgrid_build()
    off2, ids2 = o.neighbors(q)
    assert np.array_equal(off, off2) and np.array_equal(ids, ids2[:off2[-1]])
    ctx.close()


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP32_KAHAN, capi.FP64])
@pytest.mark.parametrize("grad", [False, True])
def test_many_points_equal_few_points(frame, prec, grad):
    """2^18 points or more are sorted and summed 64 to a wave, fewer a wave per point (one point per
    wave up to 4096 of them, several above): the same values bit for bit, whatever the remainders, in
    the dense cluster (several hundred passing candidates per point), off the grid and for a NaN."""
    xyz, r = frame
    s = synth.Stream(17)
    n = (1 << 18) + 3
    pick = (s.uniform(n) * len(xyz)).astype(np.int64)
    q = (xyz[pick] + s.uniform(3 * n, -3 * r, 3 * r).reshape(-1, 3)).astype(np.float32)
    q[-400:] = xyz[-400:]
    q[7] = [5.0, 0.1, 0.1]
    q[11] = [np.nan, 0.1, 0.1]
    ctx = gpu_context(xyz, r, precision=prec)
    whole = ctx.eval_points(q, grad=grad)
    for a, b in ((0, 13), (13, 4000), (4000, 4000 + 4097), (n - 20003, n)):
        part = ctx.eval_points(q[a:b], grad=grad)
        if grad:
            assert np.array_equal(whole[0][a:b], part[0]) and np.array_equal(whole[1][a:b], part[1]), (a, b)
        else:
            assert np.array_equal(whole[a:b], part), (a, b)
    ctx.close()


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP64])
def test_points_match_oracle(prec):
    """Points a wave each against the oracle, with single candidates, empty windows and more than 64
    passing candidates (a cloud of 60 particles per cell)."""
    from oracle.pyoracle import Oracle
    xyz, r = synth.random_cloud(4000, r=0.01, extent=0.16)
    xyz = np.concatenate([xyz, np.array([[0.5, 0.5, 0.5]], np.float32)])
    q = np.concatenate([xyz[::9], xyz[-1:], xyz[:50] + np.float32(0.2)]).astype(np.float32)
    ctx = gpu_context(xyz, r, precision=prec)
    f, g = ctx.eval_points(q, grad=True)
    o = Oracle(xyz, r, fp64=prec == capi.FP64)
    o.hashgrid_build()
    o.set_aniso(*ctx.aniso())
    iso = o.iso_constants()[1]
    f2, g2 = o.eval_points(q, grad=True)
    # same records, same order: FP32 rounds each term as the oracle does (libm's pow may differ by an
    # ulp per term), FP64 differs by contraction, about 1e-15 per term
    tol = 2e-6 if prec == capi.FP32 else 1e-13
    assert np.max(np.abs(f - f2)) <= tol * np.max(np.abs(iso - f2) + iso)
    assert np.max(np.abs(g - g2)) <= tol * np.max(np.abs(g2))
    ctx.close()


@pytest.mark.parametrize("prec", [capi.FP32_KAHAN, capi.FP64])
def test_many_edges_equal_few_edges(frame, prec):
    """2^16 edges or more take a thread each, fewer a wave per one to eight edges: the same vertices and counts."""
    xyz, r = frame
    s = synth.Stream(29)
    n = (1 << 16) + 5
    pick = (s.uniform(n) * len(xyz)).astype(np.int64)
    a = (xyz[pick] + s.uniform(3 * n, -2 * r, 2 * r).reshape(-1, 3)).astype(np.float32)
    b = a + np.float32(2 * r) * np.eye(3, dtype=np.float32)[np.arange(n) % 3]
    ctx = gpu_context(xyz, r, precision=prec)
    ends = np.stack([np.concatenate([p, ctx.eval_points(p)[:, None]], axis=1) for p in (a, b)], axis=1)
    ends[3] = ends[3, 0]  # no length: no step
    whole = ctx.bisect_edges(ends)
    for lo, hi in ((0, 3), (1000, 6000), (0, (1 << 16) - 1)):
        part = ctx.bisect_edges(ends[lo:hi])
        assert np.array_equal(whole[0][lo:hi], part[0], equal_nan=True) and np.array_equal(whole[1][lo:hi], part[1])
    ctx.close()


@pytest.mark.parametrize("ani,poly6", [(True, False), (False, True)])
@pytest.mark.parametrize("scene", ["sphere", "dam"])
def test_qef_vertex_values_equal_point_values(scene, ani, poly6):
    """Vertex values of leaves, by waves of nodes in the deepest levels and point by point above them."""
    xyz, r = synth.lattice_sphere(radius=0.05, r=0.005) if scene == "sphere" else synth.dam_break()
    ctx = gpu_context(xyz, r, use_ani=ani, use_poly6=poly6, qef_mode=capi.QEF_REFERENCE)
    info = ctx.run_frame()
    nodes = ctx.tree_nodes(info["n_nodes"])
    pick = (nodes["type"] == 2) & (nodes["depth"] >= info["depth_min"])
    v = nodes["node"][pick]
    f = ctx.eval_points(v[:, :3].astype(np.float32))
    ctx.close()
    assert len(v) > 1000
    assert np.array_equal(v[:, :3], v[:, :3].astype(np.float32).astype(np.float64))
    assert np.all((v[:, 3] == f) | (v[:, 3] == 0)) and np.count_nonzero(v[:, 3]) > len(v) // 4


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP32_KAHAN, capi.FP64])
@pytest.mark.parametrize("inf_factor", [4.0, 5.3, 1.0])
def test_lattice_equals_point_values(prec, inf_factor):
    """The dense lattice by waves of 4 x 4 x 4 points (cells of 4 r: one window per wave, of 5.3 r: blocks across
    cells) and a thread per point (cells of r), against the field at the same points."""
    xyz, r = synth.random_cloud(1500, r=0.01, extent=0.23)
    ctx = gpu_context(xyz, r, precision=prec)
    if inf_factor != 4.0:
        ctx.hashgrid_build(inf_factor=inf_factor)
    vals, box, sp = ctx.uniform_grid()
    nz, ny, nx = vals.shape
    f32 = np.float32
    axes = []
    for a, n in enumerate((nx, ny, nz)):
        i, st = np.arange(n), f32(n - 1)
        axes.append((f32(n - 1 - i) / st) * f32(box[2 * a]) + (i.astype(f32) / st) * f32(box[2 * a + 1]))
    z, y, x = np.meshgrid(axes[2], axes[1], axes[0], indexing="ij")
    f = ctx.eval_points(np.stack([x, y, z], axis=-1).astype(f32).reshape(-1, 3))
    ctx.close()
    assert np.array_equal(vals.reshape(-1), f.astype(f32))
