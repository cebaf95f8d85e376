"""GPU: QEF vertex values by waves of nodes, in every precision, against the same nodes swept as a mixed list, whose
vertices a wave takes one after another, and whose samples a thread each."""
import numpy as np
import pytest

from particleisosurface_amd import capi, synth
from tests.conftest import gpu_context
from tests.test_gpu_wave_sums import frame  # noqa: F401

pytestmark = pytest.mark.gpu

WAVE_NODES = 4096    # a level's nodes from which waves take them
WAVE_DENSITY = 4.0   # and its nodes, or sample points, per hash cell of 4 r


def density(nodes, depth, r, per_width):
    half = nodes["half"][nodes["depth"] == depth][0]
    return (4 * r * per_width / (2 * half)) ** 3


@pytest.mark.parametrize("prec", [capi.FP32, capi.FP32_KAHAN, capi.FP64])
@pytest.mark.parametrize("ani,poly6", [(True, False), (False, True)])
def test_vertex_values_of_a_tree_equal_those_of_a_sweep(prec, ani, poly6):
    xyz, r = synth.dam_break()
    kw = dict(precision=prec, use_ani=ani, use_poly6=poly6, qef_mode=capi.QEF_REFERENCE)
    ctx = gpu_context(xyz, r, **kw)
    info = ctx.build_tree()
    nodes = ctx.tree_nodes(info["n_nodes"])
    by_wave = 0
    for depth in range(info["depth_min"], info["n_levels"]):
        at = np.flatnonzero(nodes["depth"] == depth)
        type_, f, _, _ = ctx.sweep_level(nodes["center"][at], nodes["half"][at], nodes["depth"][at])
        leaf = type_ == capi.LEAF
        assert np.array_equal(type_, nodes["type"][at])
        assert np.array_equal(f[leaf], nodes["node"][at][leaf, 3]), depth
        if density(nodes, depth, r, 1) >= WAVE_DENSITY and len(at) >= WAVE_NODES:
            by_wave += np.count_nonzero(leaf & (f != 0))
    ctx.close()
    assert by_wave > 1000


def test_the_frame_of_the_wave_sums_has_dense_levels(frame):  # noqa: F811
    """Samples go 64 to a wave in levels of at least 4 points a hash cell and 4096 sampled nodes."""
    xyz, r = frame
    ctx = gpu_context(xyz, r)
    info = ctx.run_frame()
    nodes = ctx.tree_nodes(info["n_nodes"])
    ctx.close()
    dense = [d for d in range(info["depth_min"], info["depth_max"])
             if density(nodes, d, r, 2) >= WAVE_DENSITY
             and np.count_nonzero((nodes["depth"] == d) & (nodes["type"] != capi.EMPTY)) >= WAVE_NODES]
    assert len(dense) == 2 and dense[-1] == info["depth_max"] - 1
