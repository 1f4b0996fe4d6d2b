"""The linear query split over workgroups and lanes, and triangle tests with very
large determinants, against the oracle's one-after-another walk: bit for bit."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _soup(n, seed, span=1.0, xforms=False):
    rng = np.random.default_rng(seed)
    c = rng.random((n, 1, 3)) * span
    v = (c + 0.3 * span * rng.normal(size=(n, 3, 3))).astype(np.float32)
    s = scenes.SceneData(v, scenes.face_normals(v), np.zeros(n, np.int32),
                         scenes.make_material((0.5, 0.5, 0.5), (0.5, 0.5, 0.5), 8)[None],
                         scenes.make_lights([(2.0, 3.0, 3.0)]),
                         scenes.make_camera((0.5, 0.5, 3.0), (0.5, 0.5, 0.5), 60.0, 16, 16), 0)
    if xforms:
        s.xforms = np.stack([scenes.affine((0.2, 1.0, 0.1), 0.7, (1.1, 0.9, 1.0), (0.1, 0.0, -0.2)),
                             scenes.translation(0.3, -0.1, 0.2)])
        s.xform_index = (np.arange(n) % 3 - 1).astype(np.int32)
    return s


# rays: one, both sides of the lane split's limit (128), of a workgroup (256), many;
# triangles: one, both sides of a tile (256), several chunks
@pytest.mark.parametrize("n_rays,n_tri,xforms", [
    (1, 1, False), (1, 5000, True), (2, 257, False), (37, 1000, True), (128, 256, False), (129, 255, False),
    (256, 5000, False), (257, 700, True), (4000, 1537, False)])
def test_linear_split(n_rays, n_tri, xforms):
    from eos_amd import _lib as E
    print(f"linear n_rays={n_rays} n_tri={n_tri} xforms={xforms}", flush=True)
    s = _soup(n_tri, 11 * n_rays + n_tri, xforms=xforms)
    rng = np.random.default_rng(n_rays)
    o = (rng.random((n_rays, 3)) * 2.0 - 0.5).astype(np.float32)
    d = rng.normal(size=(n_rays, 3)).astype(np.float32)
    # every third ray starts on a triangle's first corner: a hit at t = 0 ends what the search keeps
    k = np.arange(0, n_rays, 3)
    o[k] = s.verts[(7 * k + n_tri // 3) % n_tri, 0]
    # every seventh direction is not a number: hits that lift the search's bounds
    d[np.arange(3, n_rays, 7), 1] = np.nan
    g = E.Scene(s)
    r, ref = g.trace_rays(o, d, "linear"), po.Oracle(s).nearest_linear(o, d)
    assert np.array_equal(r["hit"] == 1, ref["found"])
    assert np.array_equal(r["triangle"], ref["tri"])
    h = ref["tri"] >= 0
    assert np.array_equal(r["t"][h], ref["t"][h]) and np.array_equal(r["point"][h], ref["point"][h])
    assert np.array_equal(r["normal"][h], ref["normal"][h])


@pytest.mark.parametrize("n_rays", [64, 1000])
def test_linear_search_goes_on_after_a_hit_that_is_not_a_number(n_rays):
    """A triangle with an infinite corner hits every ray at a t that is not a
    number, in the middle of the order: hits after a t = 0 hit count again."""
    from eos_amd import _lib as E
    s = _soup(1200, 5)
    s.verts[600, 1] = np.inf
    rng = np.random.default_rng(9)
    o = s.verts[np.arange(n_rays) % 1200, 0].copy()
    o[~np.isfinite(o).all(1)] = 0.0
    d = rng.normal(size=(n_rays, 3)).astype(np.float32)
    g = E.Scene(s)
    r, ref = g.trace_rays(o, d, "linear"), po.Oracle(s).nearest_linear(o, d)
    assert np.array_equal(r["hit"] == 1, ref["found"]) and np.array_equal(r["triangle"], ref["tri"])


@pytest.mark.parametrize("span", [1.0, 1e6, 3e18, 2e19])
def test_large_determinants(span):
    """Determinants up to and beyond 2^126, where the reciprocal divides."""
    from eos_amd import _lib as E
    s = _soup(300, 3, span=span)
    rng = np.random.default_rng(4)
    o = (rng.random((500, 3)) * span).astype(np.float32)
    d = rng.normal(size=(500, 3)).astype(np.float32)
    g = E.Scene(s)
    orc = po.Oracle(s)
    r, ref = g.trace_rays(o, d, "linear"), orc.nearest_linear(o, d)
    assert np.array_equal(r["triangle"], ref["tri"])
    h = ref["tri"] >= 0
    assert h.any() or span > 1e5      # (beyond 999999 the linear search keeps nothing)
    assert np.array_equal(r["t"][h], ref["t"][h])
