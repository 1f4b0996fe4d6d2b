"""Linear searches among triangles hit at a t that is not a number (an infinite
corner): such a hit reopens a search that a hit at t = 0 has closed, wherever the
two lie in the split over chunks and lanes.  Against the oracle, bit for bit, and
no slower than a search without such triangles."""
import time

import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _soup(n, seed, bad):
    rng = np.random.default_rng(seed)
    v = (rng.random((n, 1, 3)) + 0.3 * rng.normal(size=(n, 3, 3))).astype(np.float32)
    v[bad, 1] = np.inf
    return scenes.SceneData(v, np.tile(np.float32([0, 0, 1]), (n, 3, 1)), np.zeros(n, np.int32),
                            scenes.make_material((0.5, 0.5, 0.5), (0.5, 0.5, 0.5), 8)[None],
                            scenes.make_lights([(2.0, 3.0, 3.0)]),
                            scenes.make_camera((0.5, 0.5, 3.0), (0.5, 0.5, 0.5), 60.0, 16, 16), 0)


# rays shared by 64, 16 and 2 lanes, and not; infinite corners at the ends, around
# a tile's and a slice's edges, next to each other and in every triangle of a stretch
@pytest.mark.parametrize("n_rays,n_tri", [(1, 3000), (9, 3000), (128, 3000), (129, 3000), (2000, 3000), (2000, 200)])
@pytest.mark.parametrize("bad", [[0], [-1], [255, 256, 511], [4, 8, 100, 1777], list(range(60, 160))])
def test_hits_that_are_not_numbers(n_rays, n_tri, bad):
    from eos_amd import _lib as E
    print(f"linear nan n_rays={n_rays} n_tri={n_tri} bad={bad[:4]}", flush=True)
    bad = [b % n_tri for b in bad]
    s = _soup(n_tri, n_tri + len(bad), bad)
    rng = np.random.default_rng(n_rays)
    # rays that start on corners, so that t = 0 hits close the search before and after the bad triangles
    o = s.verts[rng.integers(0, n_tri, n_rays), 0].copy()
    d = rng.normal(size=(n_rays, 3)).astype(np.float32)
    free = np.arange(n_rays) % 3 == 2
    o[free] = (rng.random((n_rays, 3)) * 2.0 - 0.5).astype(np.float32)[free]
    r, ref = E.Scene(s).trace_rays(o, d, "linear"), po.Oracle(s).nearest_linear(o, d)
    assert np.array_equal(r["hit"] == 1, ref["found"]) and np.array_equal(r["triangle"], ref["tri"])
    h = ref["tri"] >= 0
    assert np.array_equal(r["t"][h], ref["t"][h]) and np.array_equal(r["point"][h], ref["point"][h])


@pytest.mark.parametrize("n_rays,n_tri", [(4000, 13312), (300_000, 2000)])
def test_an_infinite_corner_does_not_slow_the_search(n_rays, n_tri):
    import torch
    from eos_amd import _lib as E
    g = torch.Generator(device="cuda").manual_seed(n_rays)
    o = torch.rand((n_rays, 3), generator=g, device="cuda")
    d = torch.randn((n_rays, 3), generator=g, device="cuda")
    out = torch.zeros((n_rays, 12), device="cuda")
    us = {}
    for bad in ([], [n_tri // 2]):
        sc = E.Scene(_soup(n_tri, 1, bad))
        torch.cuda.synchronize()
        runs = []
        for _ in range(6):
            t = time.perf_counter()
            sc.trace_rays_device(n_rays, o.data_ptr(), d.data_ptr(), "linear", hits_ptr=out.data_ptr())
            runs.append(1e6 * (time.perf_counter() - t))
        us[len(bad)] = min(runs[1:])
    assert us[1] < 4.0 * us[0] + 100.0, us     # a lane walking alone took 40 to 60 times as long
