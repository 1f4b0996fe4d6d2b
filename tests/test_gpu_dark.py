"""Shadow rays toward lights that add nothing to their surface are not walked:
frames equal those that walk every shadow ray (counting frames do), and the
adjoint walks them when an upstream gradient is not finite."""
import numpy as np
import pytest

from eos_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _scene(kind):
    if kind == "glass":
        s = scenes.glass(120, 90, level=3, depth=3)
    elif kind == "soup":
        s = scenes.config_b(131, 97, n=4000)
    else:
        s = scenes.config_c_dense(120, 90, nu=128, nv=64)
    # lights all around, so that many lie behind their surfaces
    rng = np.random.default_rng(2)
    p = rng.normal(size=(5, 3))
    c = s.verts.reshape(-1, 3).mean(0)
    s.lights = scenes.make_lights(c + 8.0 * p / np.linalg.norm(p, axis=1, keepdims=True), 0.2 + 0.6 * rng.random((5, 3)))
    return s


@pytest.mark.parametrize("kind", ["dense", "soup", "glass"])
@pytest.mark.parametrize("cfg", [{}, {"coop": 4, "group": 0}, {"group": 64, "group_lanes": 16}, {"steal": 0, "scatter": 0}])
def test_frames_equal_frames_that_walk_every_shadow_ray(kind, cfg):
    from eos_amd import _lib as E
    print(f"dark {kind} {cfg}", flush=True)
    s = _scene(kind)
    g = E.Scene(s)
    g.set_launch_config(**cfg)
    a = g.render(want_rgb=True, want_hits=True)
    b = g.render(want_rgb=True, want_hits=True, count_visits=True)
    assert np.array_equal(a["rgb"].view(np.uint32), b["rgb"].view(np.uint32))
    assert np.array_equal(a["rgba"], b["rgba"]) and np.array_equal(a["hit"], b["hit"])
    assert a["stats"]["shadow_rays"] == b["stats"]["shadow_rays"]
    if not cfg:
        ref = po.Oracle(s).render()
        assert np.abs(a["rgba"].astype(int) - ref["rgba"].astype(int)).max() <= 1
        imgs, _ = E.render_batch([g, g], depth=s.depth)
        assert np.array_equal(imgs[0], a["rgba"]) and np.array_equal(imgs[1], a["rgba"])


@pytest.mark.parametrize("blocked", [False, True])
@pytest.mark.parametrize("device", [False, True])
def test_infinite_upstream_gradient_on_a_surface_lit_from_behind(blocked, device):
    """Where the light behind the surface is visible, an infinite upstream gradient
    is an error (infinity times zero); where it is blocked, it is not."""
    import torch

    from eos_amd import _lib as E
    v, n = scenes.quad_grid(1, 2.0, 0.0)
    if blocked:
        w, m = scenes.quad_grid(1, 3.0, -1.0)
        v, n = np.concatenate([v, w]), np.concatenate([n, m])
    s = scenes.SceneData(v, n, np.zeros(len(v), np.int32), scenes.make_material((0.5,) * 3, (0.5,) * 3, 8)[None],
                         scenes.make_lights([(0.0, -4.0, 0.0)]),
                         scenes.make_camera((0.0, 3.0, 0.0), (0.0, 0.0, 0.0), 40.0, 8, 8, world_up=(0.0, 0.0, 1.0)), 0)
    g = E.Scene(s)
    dl = np.full((8, 8, 3), np.inf, np.float32)

    def adjoint(up):
        g.render(keep_records=True)
        if not device:
            return g.adjoint(up)[:2]
        t = torch.from_numpy(up).cuda()
        gm = torch.zeros((1, 7), dtype=torch.float64, device="cuda")
        gl = torch.zeros((1, 6), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        g.adjoint_device(s.camera, 0, t.data_ptr(), gm.data_ptr(), gl.data_ptr())
        return gm.cpu().numpy(), gl.cpu().numpy()

    gm, gl = adjoint(np.ones((8, 8, 3), np.float32))
    assert (gm == 0).all() and (gl == 0).all()
    if blocked:
        gm, gl = adjoint(dl)
        assert (gm == 0).all() and (gl == 0).all()
    else:
        with pytest.raises(E.EosError):
            adjoint(dl)
