"""torch.autograd.Function around eos_render / eos_render_adjoint (test harness).

Parameters are torch tensors on any device:
  kd, ks      [M, 3]  diffuse and specular colours
  shininess   [M]     Phong exponents (used as floats)
  light_pos   [L, 3]  point-light positions
  light_color [L, 3]  light colours
The output is the pre-quantisation image [H, W, 3] (float32, on cuda:0).
Gradients come from the hand-written HIP adjoint with hit sets held fixed
(visibility, hit points and reflection paths of the forward pass).

Each forward keeps its own materials and lights.  The scene holds one set of
hit records, so a backward whose scene was rendered or changed after its
forward (two renders in one loss, a parameter update in between) uploads its
forward's parameters again and re-traces the records instead of replaying
another call's, then puts the scene's parameters back.
"""
from __future__ import annotations

import numpy as np
import torch

from . import _lib as E


def _host_params(kd, ks, shininess, light_pos, light_color):
    """The five parameter tensors as float32 host arrays: one copy when they share a device
    (five copies, a wait each: a training step of 1M triangles 1,669 -> 1,685 us, one of a
    400 x 300 frame 662 -> 687)."""
    ts = [t.detach() for t in (kd, ks, shininess, light_pos, light_color)]
    if len({t.device for t in ts}) == 1:
        flat = torch.cat([t.to(torch.float32).reshape(-1) for t in ts]).to("cpu").numpy()
        ends = np.cumsum([t.numel() for t in ts])
        return [flat[e - t.numel():e].reshape(tuple(t.shape)) for e, t in zip(ends, ts)]
    return [t.to("cpu", torch.float32).numpy() for t in ts]


def _materials_from(base, kd, ks, shininess):
    m = base.copy()
    m["kd"][:, :3] = kd
    m["ks"][:, :3] = ks
    m["shininess"] = shininess
    return m


def _lights_from(base, pos, col):
    lt = base.copy()
    lt["position"][:, :3] = pos
    lt["position"][:, 3] = 1.0
    lt["color"][:, :3] = col
    return lt


class RenderFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, kd, ks, shininess, light_pos, light_color, scene: "E.Scene", camera, depth: int):
        h = _host_params(kd, ks, shininess, light_pos, light_color)
        mats = _materials_from(scene.data.materials, *h[:3])
        lights = _lights_from(scene.data.lights, *h[3:])
        scene.set_materials(mats)
        scene.set_lights(lights)
        W, H = int(camera["width"]), int(camera["height"])
        rgb = torch.empty((H, W, 3), dtype=torch.float32, device="cuda:0")
        torch.cuda.synchronize()
        scene.render_device(camera, depth, None, rgb_dev_ptr=rgb.data_ptr(), keep_records=True)
        ctx.scene, ctx.camera, ctx.depth = scene, camera, depth
        ctx.mats, ctx.lights = mats, lights
        ctx.generation = scene.generation   # the records this forward left on the scene
        ctx.shapes = (kd.shape[0], light_pos.shape[0])
        ctx.devices = (kd.device, light_pos.device)
        return rgb

    @staticmethod
    def backward(ctx, grad_rgb):
        scene, camera, depth = ctx.scene, ctx.camera, ctx.depth
        M, L = ctx.shapes
        g = grad_rgb.detach().to("cuda:0", torch.float32).contiguous()
        acc = torch.zeros(7 * M + 6 * max(L, 1), dtype=torch.float64, device="cuda:0")
        gm, gl = acc[:7 * M].view(M, 7), acc[7 * M:].view(-1, 6)
        torch.cuda.synchronize()
        stale = scene.generation != ctx.generation
        if stale:
            current = (scene._mats.copy(), scene._lights.copy())
            scene.set_materials(ctx.mats)
            scene.set_lights(ctx.lights)
        try:
            scene.adjoint_device(camera, depth, g.data_ptr(), gm.data_ptr(), gl.data_ptr(), recompute=stale)
        finally:
            if stale:
                scene.set_materials(current[0])
                scene.set_lights(current[1])
        gm = gm.to(ctx.devices[0], torch.float32)
        gl = gl[:L].to(ctx.devices[1], torch.float32)
        return gm[:, 0:3], gm[:, 3:6], gm[:, 6], gl[:, 0:3], gl[:, 3:6], None, None, None


def render(scene: "E.Scene", kd, ks, shininess, light_pos, light_color, camera=None, depth=None):
    camera = np.array(scene.data.camera if camera is None else camera, copy=True)
    depth = scene.data.depth if depth is None else depth
    return RenderFunction.apply(kd, ks, shininess, light_pos, light_color, scene, camera, depth)


def params_of(scene_data, device="cuda:0"):
    """(kd, ks, shininess, light_pos, light_color) tensors of a SceneData."""
    t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float32, device=device)  # noqa: E731
    return (t(scene_data.materials["kd"][:, :3]), t(scene_data.materials["ks"][:, :3]),
            t(scene_data.materials["shininess"]), t(scene_data.lights["position"][:, :3]),
            t(scene_data.lights["color"][:, :3]))
