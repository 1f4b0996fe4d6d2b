"""The reciprocal of the triangle test's determinant against correctly rounded
division: every determinant the test does not reject, and searches whose
determinants pass 2^126, where the reciprocal divides."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _scene(v):
    n = len(v)
    return scenes.SceneData(v.astype(np.float32), np.tile(np.float32([0, 0, 1]), (n, 3, 1)), np.zeros(n, np.int32),
                            scenes.make_material((0.5, 0.5, 0.5), (0.5, 0.5, 0.5), 8)[None],
                            scenes.make_lights([(2.0, 3.0, 3.0)]),
                            scenes.make_camera((0.5, 0.5, 3.0), (0.5, 0.5, 0.5), 60.0, 16, 16), 0)


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_every_determinant(sign):
    """Edges (1, 0, 0) and (0, -1, 0) at the origin and a ray from (0, 0, -+2^e) along
    +-x z: the determinant is +-x, u = v = 0 and t = 2^e times the reciprocal of
    x, exactly.  For every float x from 10^-5 (smaller determinants are rejected)."""
    import torch
    from eos_amd import _lib as E
    g = E.Scene(_scene(np.array([[[0, 0, 0], [1, 0, 0], [0, -1, 0]]])))
    n = 1 << 23
    mant = torch.arange(n, dtype=torch.int32, device="cuda")
    o, d = torch.zeros((n, 3), device="cuda"), torch.zeros((n, 3), device="cuda")
    out = torch.zeros((n, 12), device="cuda")
    for e in range(-17, 128):
        if e % 16 == 0:
            print(f"determinants sign={sign} exponent={e}", flush=True)
        x = (mant + ((e + 127) << 23)).view(torch.float32)
        o[:, 2] = -sign * 2.0**e
        d[:, 2] = sign * x
        torch.cuda.synchronize()
        g.trace_rays_device(n, o.data_ptr(), d.data_ptr(), "linear", hits_ptr=out.data_ptr())
        if e < 126:
            # 1 / x is not within 2^-49 of half way between two floats, so rounding twice rounds correctly
            want = ((1.0 / x.double()).float() * 2.0**e)
        else:
            want = torch.from_numpy(np.float32(1.0) / x.cpu().numpy() * np.float32(2.0**e)).cuda()
        hit = x >= torch.tensor(0.00001, dtype=torch.float32, device="cuda")
        assert torch.equal(out[:, 3].view(torch.int32) == 1, hit), e
        assert torch.equal(out[hit, 8].view(torch.int32), want[hit].view(torch.int32)), e


@pytest.mark.parametrize("span,length", [(1e9, 1e20), (1e12, 1e14), (3e9, 2e19)])
def test_searches_beyond_2_126(span, length):
    """Long directions: determinants around and beyond 2^126 at distances a search keeps."""
    from eos_amd import _lib as E
    rng = np.random.default_rng(4)
    c = rng.random((300, 1, 3)) * span
    s = _scene(c + 0.3 * span * rng.normal(size=(300, 3, 3)))
    o = (rng.random((500, 3)) * span).astype(np.float32)
    d = (rng.normal(size=(500, 3)) * length).astype(np.float32)
    v = s.verts.astype(np.float64)
    det = np.abs(np.einsum("tk,rtk->rt", v[:, 1] - v[:, 0], np.cross(d[:, None].astype(np.float64), v[:, 2] - v[:, 0])))
    r, ref = E.Scene(s).trace_rays(o, d, "linear"), po.Oracle(s).nearest_linear(o, d)
    h = ref["tri"] >= 0
    kept = det[np.nonzero(h)[0], ref["tri"][h]]
    assert h.sum() > 300 and (kept >= 2.0**126).sum() > 50 and (kept < 2.0**126).sum() > 50
    assert np.array_equal(r["hit"] == 1, ref["found"]) and np.array_equal(r["triangle"], ref["tri"])
    assert np.array_equal(r["t"][h], ref["t"][h])
