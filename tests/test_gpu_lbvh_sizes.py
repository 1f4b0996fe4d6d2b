"""The LBVH at the sizes where its kernels' tiles end: waves of the sort (64 keys),
its workgroups (1,024), the box pyramid's blocks (1,024 leaves) and upper levels,
the node numbering's workgroups (256), and the largest trees a leaf size gives."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _u32(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("leaf_max", [1, 3])
@pytest.mark.parametrize("n", [1, 3, 4, 63, 65, 256, 257, 258, 513, 1023, 1024, 1025, 2049, 4097, 66000])
def test_lbvh_at_tile_edges(n, leaf_max):
    from eos_amd import _lib as E
    print(f"lbvh n={n} leaf_max={leaf_max}", flush=True)
    s = scenes.config_b(16, 16, n=n)
    if n % 2:        # half the triangles on top of one another: equal codes
        s.verts[n // 2:] = s.verts[:1]
    g = E.Scene(s, leaf_max=leaf_max)
    ref = po.lbvh_build(s.verts, leaf_max)
    assert np.array_equal(g.debug_read("morton_sorted"), ref["codes"]) and np.array_equal(g.debug_read("perm"), ref["perm"])
    assert g.build_stats["num_nodes4"] == len(ref["nodes4"])
    if len(ref["nodes4"]):
        assert np.array_equal(_u32(g.debug_read("nodes4"))[:, :28], _u32(ref["nodes4"])[:, :28])
    assert np.array_equal(_u32(g.debug_read("tris"))[:, :11], _u32(ref["tris"])[:, :11])
    if n > 1:
        assert np.array_equal(_u32(g.debug_read("ibox")), _u32(ref["ibox"]))
        assert np.array_equal(g.debug_read("kparent"), ref["kparent"])
    # built again in the same buffers
    g.build(leaf_max)
    assert np.array_equal(g.debug_read("perm"), ref["perm"])


def test_deepest_trees_fit():
    """Triangles whose centroids halve their distance to a corner: chains, the trees
    with the most 4-wide nodes per triangle."""
    from eos_amd import _lib as E
    n = 200
    c = np.zeros((n, 3))
    c[:, 0] = 0.5 ** (np.arange(n) % 10)
    c[:, 1] = 0.5 ** (np.arange(n) // 10 % 10)
    c[:, 2] = 0.5 ** (np.arange(n) // 100)
    v = (c[:, None, :] + 1e-4 * np.eye(3)[None]).astype(np.float32)
    s = scenes.config_b(16, 16, n=n)
    s.verts[:] = v
    for leaf_max in (1, 2, 3, 4, 8):
        g = E.Scene(s, leaf_max=leaf_max)
        ref = po.lbvh_build(s.verts, leaf_max)
        assert g.build_stats["num_nodes4"] == len(ref["nodes4"])
        assert np.array_equal(_u32(g.debug_read("nodes4"))[:, :28], _u32(ref["nodes4"])[:, :28])
