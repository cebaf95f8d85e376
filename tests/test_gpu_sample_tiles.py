"""GPU: samples merged per tile of nodes, and over the whole level, against one thread per sample, bit for bit."""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context

pytestmark = pytest.mark.gpu


def spread():
    """Particles alone and in pairs: tiles whose nodes lie far apart (cells of a tile's box exceed the buckets)."""
    xyz, r = synth.random_cloud(700, r=0.01, extent=3.0)
    return np.concatenate([xyz, xyz[:90] + np.float32(0.4 * r)]), r


FRAMES = {
    "one": lambda: (np.array([[0.1, 0.2, 0.3], [0.104, 0.2, 0.3], [0.1, 0.205, 0.3]], np.float32), 0.01),  # one tile
    "sphere": lambda: synth.lattice_sphere(radius=0.05, r=0.005),   # a few tiles, points by waves of their own
    "spread": spread,
    "dam": synth.dam_break,                                         # deepest level 64 to a wave, the others not
    "crown": lambda: synth.crown_splash(pool_layers=6, n_drops=20000),  # D_min merged over the level
}


@pytest.mark.parametrize("name,prec,qef", [
    ("one", capi.FP32, 0), ("one", capi.FP64, capi.QEF_REFERENCE),
    ("sphere", capi.FP32_KAHAN, 0), ("sphere", capi.FP64, capi.QEF_SVD64),
    ("spread", capi.FP32, capi.QEF_REFERENCE), ("spread", capi.FP32_KAHAN, 0),
    ("dam", capi.FP32, 0), ("dam", capi.FP64, capi.QEF_REFERENCE),
    ("crown", capi.FP32_KAHAN, 0),
])
def test_merged_samples_equal_single_samples(name, prec, qef):
    xyz, r = FRAMES[name]()
    out = []
    for dedupe in (True, False):
        ctx = gpu_context(xyz, r, precision=prec, qef_mode=qef, sample_dedupe=dedupe)
        info = ctx.run_frame()
        out.append((info, ctx.tree_nodes(info["n_nodes"]), ctx.mesh(), ctx.stats()))
        ctx.close()
    (ia, na, ma, sa), (ib, nb, mb, sb) = out
    assert ia == ib
    for key in ("type", "id", "depth", "child", "node"):
        assert np.array_equal(na[key], nb[key]), key
    assert np.array_equal(ma[0], mb[0]) and np.array_equal(ma[1], mb[1])
    assert sa["field_evals"] == sb["field_evals"] and sa["sample_evals"] == sb["sample_evals"]
    if name == "crown":  # more nodes than go by tiles at a point per cell
        assert np.count_nonzero(na["depth"] == ia["depth_min"]) > 1 << 15


@pytest.mark.parametrize("prec,qef", [(capi.FP32_KAHAN, 0), (capi.FP64, capi.QEF_REFERENCE)])
def test_tree_with_the_normals_it_reads(prec, qef):
    """From 2^20 particles on a tree takes the normals of the cells that its curvatures read; the same tree as
    with every normal there before."""
    xyz, r = FRAMES["crown"]()
    assert len(xyz) >= 1 << 20
    out = []
    for before in (False, True):
        ctx = gpu_context(xyz, r, precision=prec, qef_mode=qef)
        if before:
            ctx.particle_normals()
        info = ctx.build_tree()
        out.append((info, ctx.tree_nodes(info["n_nodes"]), ctx.stats()["grad_evals"]))
        ctx.close()
    (ia, na, ga), (ib, nb, gb) = out
    assert ia["n_nodes"] == ib["n_nodes"] and ga == gb
    for key in ("type", "id", "depth", "child", "node"):
        assert np.array_equal(na[key], nb[key]), key
