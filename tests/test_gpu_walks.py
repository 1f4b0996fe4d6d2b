"""Ray queries at the launch sizes where the walk changes (a wave per ray, 16 lanes
per ray, a lane per ray), and a tree past 4 GiB, which takes the kernels with 64-bit
addresses."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xforms", [False, True])
def test_queries_at_the_walks_limits(xforms):
    from eos_amd import _lib as E
    s = scenes.config_f(32, 32, instances=6, nu=48, nv=24) if xforms else scenes.config_b(32, 32, n=30000)
    rng = np.random.default_rng(1)
    n = 400_000                      # a lane per ray, several rays per lane
    lo, hi = s.verts.min((0, 1)) - 1.0, s.verts.max((0, 1)) + 1.0
    o = (lo + (hi - lo) * rng.random((n, 3))).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    g = E.Scene(s)
    ref, occ = g.trace_rays(o, d, "nearest"), g.trace_rays(o, d, "occluded")
    b = po.Oracle(s).nearest(o[:3000], d[:3000])
    assert np.array_equal(ref["triangle"][:3000], b["tri"])
    for k in (1, 2, 3, 2559, 2560, 2561, 20479, 20480, 20481, 50_000):
        print(f"walks xforms={xforms} rays={k}", flush=True)
        assert g.trace_rays(o[-k:], d[-k:], "nearest").tobytes() == ref[-k:].tobytes()
        assert np.array_equal(g.trace_rays(o[-k:], d[-k:], "occluded"), occ[-k:])


def test_a_tree_past_4_gib():
    import torch

    from eos_amd import _lib as E
    n = 50_000_000
    free, _ = torch.cuda.mem_get_info()
    if free < 40 << 30:
        pytest.skip("needs 40 GiB of device memory")
    rng = np.random.default_rng(7)
    verts = np.empty((n, 3, 3), np.float32)
    verts[:] = rng.random((n, 1, 3), dtype=np.float32)
    verts[:, 1, 0] += 0.004
    verts[:, 2, 1] += 0.004
    # a few large ones, so that most rays hit something far in the arrays too
    verts[-2000:] += 0.1 * rng.normal(size=(2000, 3, 3)).astype(np.float32)
    normals = np.zeros_like(verts)
    normals[:, :, 2] = 1.0
    s = scenes.SceneData(verts, normals, np.zeros(n, np.int32),
                         scenes.make_material((0.5,) * 3, (0.2,) * 3, 8, 0.3, True)[None],
                         scenes.make_lights([(2.0, 3.0, 3.0)]),
                         scenes.make_camera((0.5, 0.5, 2.6), (0.5, 0.5, 0.5), 40.0, 64, 48), 1)
    g = E.Scene(s, leaf_max=1)     # the most nodes per triangle
    assert 48 * n + 128 * g.build_stats["num_nodes4"] > 1 << 32
    print(f"tree past 4 GiB: {g.build_stats['num_nodes4']} nodes", flush=True)
    o = rng.random((300, 3)).astype(np.float32)
    d = rng.normal(size=(300, 3)).astype(np.float32)
    near, lin = g.trace_rays(o, d, "nearest"), g.trace_rays(o, d, "linear")
    assert (near["triangle"] >= 0).sum() > 250
    assert np.array_equal(near["triangle"], lin["triangle"]) and np.array_equal(near["t"], lin["t"])
    assert np.array_equal(g.trace_rays(o, d, "occluded"), near["triangle"] >= 0)
    a, b = g.render(want_hits=True), g.render(want_hits=True, count_visits=True)
    assert np.array_equal(a["rgba"], b["rgba"]) and np.array_equal(a["hit"], b["hit"])
    assert (a["hit"] >= 0).any()
