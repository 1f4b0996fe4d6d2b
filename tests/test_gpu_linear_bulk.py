"""Linear queries of more rays than one scratch array holds runs for: a scanning
workgroup answers its rays itself.  Against the oracle, bit for bit."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _soup(n, seed):
    rng = np.random.default_rng(seed)
    v = (rng.random((n, 1, 3)) + 0.3 * rng.normal(size=(n, 3, 3))).astype(np.float32)
    s = scenes.SceneData(v, scenes.face_normals(v), np.zeros(n, np.int32),
                         scenes.make_material((0.5, 0.5, 0.5), (0.5, 0.5, 0.5), 8)[None],
                         scenes.make_lights([(2.0, 3.0, 3.0)]),
                         scenes.make_camera((0.5, 0.5, 3.0), (0.5, 0.5, 0.5), 60.0, 16, 16), 0)
    s.xforms = np.stack([scenes.affine((0.2, 1.0, 0.1), 0.7, (1.1, 0.9, 1.0), (0.1, 0.0, -0.2))])
    s.xform_index = (np.arange(n) % 2 - 1).astype(np.int32)
    return s


# one triangle tile and several; just above the rays of the fixed scratch array,
# and fewer rays that still get one chunk
@pytest.mark.parametrize("n_rays,n_tri", [((1 << 20) + 257, 130), (600_001, 600)])
def test_one_chunk_answers_its_rays(n_rays, n_tri):
    from eos_amd import _lib as E
    print(f"linear bulk n_rays={n_rays} n_tri={n_tri}", flush=True)
    s = _soup(n_tri, n_tri)
    rng = np.random.default_rng(n_rays)
    o = (rng.random((n_rays, 3)) * 2.0 - 0.5).astype(np.float32)
    d = rng.normal(size=(n_rays, 3)).astype(np.float32)
    k = np.arange(0, n_rays, 3)
    o[k] = s.verts[(7 * k) % n_tri, 0]
    d[np.arange(3, n_rays, 7), 1] = np.nan
    r, ref = E.Scene(s).trace_rays(o, d, "linear"), po.Oracle(s).nearest_linear(o, d)
    assert np.array_equal(r["hit"] == 1, ref["found"]) and np.array_equal(r["triangle"], ref["tri"])
    h = ref["tri"] >= 0
    assert h.sum() > n_rays // 20
    for a, b in (("t", "t"), ("point", "point"), ("normal", "normal")):
        assert np.array_equal(r[a][h], ref[b][h]), a
