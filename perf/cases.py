"""Timed workloads of the render path, each one pass through public entry points.

``listed`` names the workloads, ``draw`` makes more of the same ranges,
``prepare`` builds what a program holds before the call (scene with its LBVH,
cameras, rays, output buffers on the GPU), ``run`` is one pass, ``work`` the
bytes and operations a pass cannot do without, ``exact`` the 64-bit answer
where a brute-force search is affordable.

Kinds of passes:
  frame    one eos_render of a camera into a device image
  frames   eos_render_frames, a camera path with two frames in flight
  batch    eos_render_batch, many small scenes in one frame
  query    eos_trace_rays: caller-given rays against a scene
  train    autograd.render and its backward: image and parameter gradients
  moving   a scene whose instances move: transforms set, LBVH rebuilt, frame rendered
"""
from __future__ import annotations

import math

import numpy as np
import torch

from eos_amd import _lib as E
from eos_amd import autograd as G
from eos_amd import scenes as S


def listed():
    return [
        # a thumbnail or a unit test's frame: a small scene, few pixels; launches and latency
        {"name": "thumbnail", "kind": "frame", "scene": "plane", "tris": 13312, "width": 256, "height": 256,
         "lights": 1, "depth": 1, "aa": 1},
        # the viewer's frame: one scanned mesh of 70k triangles placed by a transformation, 720p, two
        # lights, the renderers' default depth of 4
        {"name": "viewer_720p", "kind": "frame", "scene": "placed", "tris": 69696, "width": 1280, "height": 720,
         "lights": 2, "depth": 4, "aa": 1},
        # the still frame at full size: 4.2M triangles, 4K, four lights, reflections
        {"name": "frame_4k", "kind": "frame", "scene": "sphere", "tris": 4194304, "width": 3840, "height": 2160,
         "lights": 4, "depth": 3, "aa": 1},
        # transparent materials (ray trees), anti-aliased, an odd image size
        {"name": "glass_aa", "kind": "frame", "scene": "glass", "tris": 16512, "width": 1365, "height": 767,
         "lights": 2, "depth": 3, "aa": 2},
        # a camera flying close over a mesh: most rays hit, shadows and reflections dominate
        {"name": "flight_1080p", "kind": "frames", "scene": "close", "tris": 1048576, "width": 1920, "height": 1080,
         "lights": 4, "depth": 3, "frames": 4},
        # a data generator's batch: many small random scenes in one captured frame
        {"name": "batch_16", "kind": "batch", "scenes": 16, "tris": 60000, "width": 512, "height": 512, "lights": 2,
         "depth": 2},
        # picking and line of sight from host code: a few rays, host arrays
        {"name": "pick_rays", "kind": "query", "scene": "placed", "tris": 69696, "mode": "nearest", "rays": 1000,
         "host": True},
        # a simulation's bulk queries: incoherent rays, nearest hits, device arrays
        {"name": "nearest_rays", "kind": "query", "scene": "sphere", "tris": 1048576, "mode": "nearest",
         "rays": 1000003, "host": False},
        # bulk visibility between points inside a cloud of triangles
        {"name": "occluded_rays", "kind": "query", "scene": "soup", "tris": 400000, "mode": "occluded",
         "rays": 500000, "host": False},
        # the search without a hierarchy (the driver's useBvh(false) route, and the checker of the others)
        {"name": "linear_rays", "kind": "query", "scene": "plane", "tris": 13312, "mode": "linear", "rays": 4000,
         "host": False},
        # one optimisation step: image, then gradients of 256 materials and 8 lights
        {"name": "train_step", "kind": "train", "scene": "sphere", "tris": 1000000, "width": 1024, "height": 1024,
         "lights": 8, "materials": 256, "depth": 2},
        # an animation's frame: 64 instances move, the tree is rebuilt, a 540p frame is rendered
        {"name": "moving_540p", "kind": "moving", "scene": "instances", "tris": 1050624, "width": 960, "height": 540,
         "lights": 2, "depth": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frames", "batch", "query", "query", "query", "train", "moving"])
    w = _log_int(rng, 200, 2600)
    h = max(64, int(w * rng.uniform(0.5, 1.0)))
    if kind == "frame":
        scene = rng.choice(["plane", "placed", "sphere", "close", "soup", "glass"])
        c = {"kind": kind, "scene": scene, "tris": _log_int(rng, 5000, 1000000), "width": w, "height": h,
             "lights": rng.randint(1, 6), "depth": rng.randint(0, 4), "aa": rng.choice([1, 1, 1, 2])}
        if scene in ("close", "soup", "glass") or c["aa"] > 1:      # no costlier than the largest listed frame
            s = min(1.0, math.sqrt(1.0e6 / (w * h)))
            c["width"], c["height"] = max(64, int(w * s)), max(64, int(h * s))
            c["depth"] = min(c["depth"], 3)
        return c
    if kind == "frames":
        return {"kind": kind, "scene": rng.choice(["placed", "sphere", "close"]), "tris": _log_int(rng, 20000, 1000000),
                "width": min(w, 1920), "height": min(h, 1080), "lights": rng.randint(1, 4), "depth": rng.randint(0, 3),
                "frames": rng.randint(2, 4)}
    if kind == "batch":
        r = rng.choice([129, 256, 384, 512])
        return {"kind": kind, "scenes": rng.randint(3, 16), "tris": _log_int(rng, 5000, 60000), "width": r,
                "height": r, "lights": rng.randint(1, 2), "depth": rng.randint(0, 2)}
    if kind == "query":
        mode = rng.choice(["nearest", "occluded", "linear"])
        if mode == "linear":
            return {"kind": kind, "scene": rng.choice(["plane", "soup"]), "tris": _log_int(rng, 500, 40000),
                    "mode": mode, "rays": _log_int(rng, 1, 20000), "host": False}
        rays = _log_int(rng, 1, 1000000)
        return {"kind": kind, "scene": rng.choice(["placed", "sphere", "soup", "plane"]),
                "tris": _log_int(rng, 5000, 1000000), "mode": mode, "rays": rays, "host": rays <= 20000}
    if kind == "train":
        r = _log_int(rng, 400, 1024)
        return {"kind": kind, "scene": rng.choice(["sphere", "close"]), "tris": _log_int(rng, 100000, 1000000),
                "width": r, "height": max(300, int(r * rng.uniform(0.6, 1.0))), "lights": rng.randint(1, 8),
                "materials": _log_int(rng, 1, 256), "depth": rng.randint(0, 2)}
    return {"kind": kind, "scene": "instances", "tris": _log_int(rng, 20000, 1050000), "width": min(w, 960),
            "height": min(h, 540), "lights": rng.randint(1, 3), "depth": rng.randint(0, 2)}


# ---------------------------------------------------------------- scenes

def _materials(rng, m, reflective=True):
    kd, ks = 0.1 + 0.8 * rng.uniform(3 * m).reshape(m, 3), 0.1 + 0.8 * rng.uniform(3 * m).reshape(m, 3)
    sh, rf = np.rint(4.0 + 124.0 * rng.uniform(m)), 0.1 + 0.4 * rng.uniform(m)
    return np.stack([S.make_material(kd[i], ks[i], sh[i], rf[i], reflective) for i in range(m)])


def _lights(rng, k, radius, center=(0.0, 0.0, 0.0)):
    d = rng.normal(3 * k).reshape(k, 3)
    d[:, 1:] = np.abs(d[:, 1:]) + (0.2, 0.0)          # above, towards the camera
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return S.make_lights(np.asarray(center) + radius * d, 0.4 + 0.5 * rng.uniform(3 * k).reshape(k, 3))


def _grid(tris, per=2):
    """nu, nv of a UV sphere of about `tris` triangles (nu = 2 nv)."""
    nv = max(8, int(round(math.sqrt(tris / (2.0 * per)))))
    return 2 * nv, nv


def _jitter(rng, eye, amount):
    return np.asarray(eye, np.float64) + amount * (2.0 * rng.uniform(3) - 1.0)


def _scene(case, seed, tris=None):
    """The case's scene, its shape, materials, lights and camera all made from the seed."""
    rng = S.Rng(0x9E37 + 7919 * seed)
    kind, n = case.get("scene", "soup"), tris or case["tris"]
    w, h = case.get("width", 64), case.get("height", 64)
    nl, depth = case.get("lights", 1), case.get("depth", 0)
    if kind == "plane":                               # icosphere over a ground plane
        cells = max(4, int(round(math.sqrt(max(n - 5120, n // 2) / 2.0))))
        sv, sn = S.icosphere(4 if n >= 10240 else (3 if n >= 2560 else 2))
        pv, pn = S.quad_grid(cells, 5.0, -1.0)
        mat = np.concatenate([np.zeros(len(sv), np.int32), np.ones(len(pv), np.int32)])
        mats = np.concatenate([_materials(rng, 1), S.make_material((0.7, 0.7, 0.7), (0.0, 0.0, 0.0), 32)[None]])
        lights = _lights(rng, nl, 5.0)
        cam = S.make_camera(_jitter(rng, (0.0, 1.0, 4.0), 0.3), (0.0, 0.0, 0.0), 60.0, w, h)
        return S.SceneData(np.concatenate([sv, pv]), np.concatenate([sn, pn]), mat, mats, lights, cam, depth)
    if kind == "soup":                                # random triangles in the unit cube
        v, nn = S.soup(n, seed, sigma_median=0.004 * math.sqrt(1e6 / n))
        lights = _lights(rng, nl, 3.0, (0.5, 0.5, 0.5))
        d = _jitter(rng, (0.0, 0.2, 1.0), 0.5)
        cam = S.make_camera(np.array([0.5, 0.5, 0.5]) + 2.2 * d / np.linalg.norm(d), (0.5, 0.5, 0.5), 60.0, w, h)
        return S.SceneData(v, nn, np.zeros(n, np.int32), _materials(rng, 1), lights, cam, depth)
    if kind == "glass":                               # glass, water-and-mirror and mirror spheres over a plane
        s = S.glass(w, h, level=max(2, min(5, int(round(math.log(max(n, 100) / 60.0, 4))))), depth=depth)
        s.camera = S.make_camera(_jitter(rng, (0.0, 0.9, 3.6), 0.3), (0.0, -0.1, 0.0), 55.0, w, h)
        s.lights = _lights(rng, nl, 4.5)
        return s
    nu, nv = _grid(n)
    if kind == "instances":                           # 64 copies of one mesh over a plane
        nu, nv = _grid(max(n - 2048, 64 * 256) / 64.0)
        sv, sn, _ = S.displaced_sphere(nu, nv, seed)
        pv, pn = S.quad_grid(32, 18.0, -1.4)
        xi = np.concatenate([np.repeat(np.arange(64, dtype=np.int32), len(sv)), np.full(len(pv), -1, np.int32)])
        mat = np.concatenate([np.repeat(np.arange(64, dtype=np.int32) % 8, len(sv)), np.full(len(pv), 8, np.int32)])
        mats = np.concatenate([_materials(rng, 8), S.make_material((0.6, 0.6, 0.6), (0.1, 0.1, 0.1), 8)[None]])
        cam = S.make_camera(_jitter(rng, (0.0, 7.0, 13.0), 0.5), (0.0, -0.4, 1.0), 60.0, w, h)
        return S.SceneData(np.concatenate([np.tile(sv, (64, 1, 1)), pv]), np.concatenate([np.tile(sn, (64, 1, 1)), pn]),
                           mat, mats, _lights(rng, nl, 24.0), cam, depth, xforms=_places(rng, 0.0), xform_index=xi)
    v, nn, radius = S.displaced_sphere(nu, nv, seed)
    m = case.get("materials", 16)
    lo, hi = float(radius.min()), float(radius.max())
    mat = np.clip(((radius - lo) / max(hi - lo, 1e-30) * m).astype(np.int32), 0, m - 1)
    if kind == "close":                               # the mesh fills the frame
        v = (v * np.float32(4.0)).astype(np.float32)
        d = _jitter(rng, (0.3, 0.45, 1.0), 0.2)
        cam = S.make_camera(5.8 * d / np.linalg.norm(d), (0.0, 0.0, 0.0), 60.0, w, h)
        return S.SceneData(v, nn, mat, _materials(rng, m), _lights(rng, nl, 16.0), cam, depth)
    if kind == "placed":                              # one mesh placed by a transformation, as an OBJ model is
        cam = S.make_camera(_jitter(rng, (2.0, 0.0, 3.0), 0.2), (2.0, -1.0, -2.0), 60.0, w, h)
        return S.SceneData(v, nn, np.zeros(len(v), np.int32), _materials(rng, 1, False), _lights(rng, nl, 24.0), cam,
                           depth, xforms=S.translation(2.0, -1.0, -2.0)[None], xform_index=np.zeros(len(v), np.int32))
    cam = S.make_camera(_jitter(rng, (0.0, 0.4, 3.3), 0.2), (0.0, 0.0, 0.0), 60.0, w, h)
    return S.SceneData(v, nn, mat, _materials(rng, m), _lights(rng, nl, 4.0), cam, depth)


def _places(rng, phase):
    """64 placements on an 8 x 8 grid: rotation, scale, height."""
    u = rng.uniform(64 * 4).reshape(64, 4)
    return np.stack([S.affine((u[k, 0] - 0.5, 1.0, u[k, 1] - 0.5), 6.0 * u[k, 2] + phase, [0.6 + 0.6 * u[k, 3]] * 3,
                              ((k % 8 - 3.5) * 2.6, 0.2 * u[k, 0], (3.5 - k // 8) * 2.6)) for k in range(64)])


def _rays(case, data, seed):
    """Origins around and inside the scene, directions towards points of its bounding box."""
    rng = S.Rng(0xABCD + 104729 * seed)
    n = case["rays"]
    v = data.verts.reshape(-1, 3).astype(np.float64)
    if data.xforms is not None:
        v = v + data.xforms[0].reshape(4, 4)[3, :3]
    lo, hi = v.min(0), v.max(0)
    c, half = 0.5 * (lo + hi), 0.5 * (hi - lo) + 1e-3
    o = c + 1.6 * half * (2.0 * rng.uniform(3 * n).reshape(n, 3) - 1.0)
    t = c + 0.9 * half * (2.0 * rng.uniform(3 * n).reshape(n, 3) - 1.0)
    d = t - o
    d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-9)
    return o.astype(np.float32), d.astype(np.float32)


# ---------------------------------------------------------------- passes

def _device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _image(case):
    return torch.zeros((case["height"], case["width"], 4), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "batch":
        # triangle counts spread around the case's, as a generator's scenes differ
        sizes = [max(16, int(case["tris"] * (0.3 + 1.4 * (k + 0.5) / case["scenes"]))) for k in range(case["scenes"])]
        st["scenes"] = [E.Scene(_scene(case, 1000 * seed + k, n), build=False) for k, n in enumerate(sizes)]
        E.build_batch(st["scenes"])
        st["out"] = [_image(case) for _ in sizes]
        st["ptrs"] = [t.data_ptr() for t in st["out"]]
        torch.cuda.synchronize()
        return st
    data = _scene(case, seed)
    st["scene"] = sc = E.Scene(data)
    if kind in ("frame", "moving"):
        st["out"] = _image(case)
        if kind == "moving":
            # the instances' places at the animation's next moment (one moment per state: passes compare)
            st["places"], st["index"] = _places(S.Rng(31 + seed), 0.3), data.xform_index
    elif kind == "frames":
        rng = S.Rng(17 + seed)
        eye, up = data.camera["position"].astype(np.float64), float(np.linalg.norm(data.camera["view"]))
        st["cams"] = np.stack([S.make_camera(eye + 0.02 * k * (rng.uniform(3) - 0.5) * up, (0.0, 0.0, 0.0), 60.0,
                                             case["width"], case["height"]) for k in range(case["frames"])])
        st["out"] = [_image(case) for _ in range(case["frames"])]
        st["ptrs"] = [t.data_ptr() for t in st["out"]]
    elif kind == "query":
        o, d = _rays(case, data, seed)
        st["o"], st["d"] = (o, d) if case["host"] else (_device(o), _device(d))
        if not case["host"]:
            n = case["rays"]
            st["out"] = (torch.zeros(n, dtype=torch.uint8, device="cuda") if case["mode"] == "occluded"
                         else torch.zeros((n, 12), dtype=torch.float32, device="cuda"))
    elif kind == "train":
        st["params"] = [p.requires_grad_() for p in G.params_of(data)]
        g = torch.Generator(device="cuda").manual_seed(seed)
        st["grad"] = torch.randn((case["height"], case["width"], 3), generator=g, device="cuda")
    torch.cuda.synchronize()
    st["camera"], st["depth"] = data.camera, sc.data.depth
    return st


def _hit_fields(rec):
    """An RAY_HIT record's fields: floats (point, normal, t u v) and integers (hit, material, triangle)."""
    if isinstance(rec, np.ndarray):
        return {"point": rec["point"], "normal": rec["normal"], "tuv": np.stack([rec["t"], rec["u"], rec["v"]], 1),
                "ids": np.stack([rec["hit"], rec["material"], rec["triangle"]], 1)}
    return {"point": rec[:, 0:3], "normal": rec[:, 4:7], "tuv": rec[:, 8:11],
            "ids": rec.view(torch.int32)[:, 3::4]}


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "frame":
        st["scene"].render_device(st["camera"], st["depth"], st["out"].data_ptr(),
                                  aa_samples=case["aa"] if case["aa"] > 1 else 0)
        return st["out"]
    if kind == "frames":
        st["scene"].render_frames(st["cams"], st["ptrs"], depth=st["depth"])
        return st["out"]
    if kind == "batch":
        E.render_batch(st["scenes"], depth=case["depth"], use_graph=True, device_ptrs=st["ptrs"])
        return st["out"]
    if kind == "query":
        sc, mode = st["scene"], case["mode"]
        if case["host"]:
            out = sc.trace_rays(st["o"], st["d"], mode)
            return out if mode == "occluded" else _hit_fields(out)
        occ = mode == "occluded"
        sc.trace_rays_device(case["rays"], st["o"].data_ptr(), st["d"].data_ptr(), mode,
                             None if occ else st["out"].data_ptr(), st["out"].data_ptr() if occ else None)
        return st["out"] if occ else _hit_fields(st["out"])
    if kind == "train":
        for p in st["params"]:
            p.grad = None
        rgb = G.render(st["scene"], *st["params"], camera=st["camera"], depth=st["depth"])
        rgb.backward(st["grad"])
        return [rgb.detach()] + [p.grad for p in st["params"]]
    sc = st["scene"]
    sc.set_transforms(st["places"], st["index"])
    sc.build()
    sc.render_device(st["camera"], st["depth"], st["out"].data_ptr())
    return st["out"]


def work(case):
    """Inputs read once and outputs written once; per primary ray one box test of four children per tree
    level and one triangle test.  Which shadow and reflection rays follow is the scene's affair: not counted."""
    kind = case["kind"]
    tri_ops, node_ops = 50, 48
    n = case["tris"] * (case["scenes"] if kind == "batch" else 1)
    levels = max(1.0, math.log(max(case["tris"], 4) / 4.0, 4))
    if kind == "query":
        out = 1 if case["mode"] == "occluded" else 48
        per_ray = case["tris"] * tri_ops if case["mode"] == "linear" else levels * node_ops + tri_ops
        # nearest and linear: geometry and the hit's normals; each triangle at most once, at most what rays reach
        touched = n if case["mode"] == "linear" else min(n, 8 * case["rays"])
        return {"bytes": 36 * touched + (24 + out) * case["rays"], "flops": per_ray * case["rays"]}
    images = case.get("frames", 1) * (case["scenes"] if kind == "batch" else 1)
    pix = case["width"] * case["height"] * images
    rays = pix * case.get("aa", 1) ** 2
    # triangles a frame reaches: each at most once, at most one per ray
    b = 36 * min(n, rays) + 4 * pix
    if kind == "train":
        b += 12 * pix * 2 + 72 * (case["materials"] + case["lights"])
    if kind == "moving":
        b += n * (72 + 8 + 96)                        # input triangles read, triangle records written
    return {"bytes": b, "flops": rays * (levels * node_ops + tri_ops)}


# ---------------------------------------------------------------- 64-bit answers

def exact(case, seed):
    """Nearest hits by a brute-force search in 64 bits where rays times triangles allow it.  Images are
    bytes (no value here); a training step's 64-bit answer would take minutes: None."""
    if case["kind"] != "query" or case["mode"] == "occluded" or case["rays"] * case["tris"] > 1.0e9:
        return None
    data = _scene(case, seed)
    o, d = (_device(a).double() for a in _rays(case, data, seed))
    v, nn = _device(data.verts).double(), _device(data.normals).double()
    if data.xforms is not None:                       # "placed": one translation for all triangles
        v = v + _device(data.xforms[0].reshape(4, 4)[3, :3]).double()
    e1, e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    n, step = case["rays"], max(1, 20_000_000 // len(v))
    best = [torch.zeros(n, k, dtype=torch.float64, device="cuda") for k in (3, 3, 3)]
    for a in range(0, n, step):
        b = min(n, a + step)
        O, D = o[a:b, None], d[a:b, None]
        P = torch.linalg.cross(D, e2[None].expand(b - a, -1, -1))
        det = (e1[None] * P).sum(-1)
        T = O - v[None, :, 0]
        Q = torch.linalg.cross(T, e1[None].expand(b - a, -1, -1))
        inv = 1.0 / det
        t, u, w = (e2[None] * Q).sum(-1) * inv, (T * P).sum(-1) * inv, (D * Q).sum(-1) * inv
        ok = (det.abs() >= 1e-5) & (t >= 0) & (u >= 0) & (w >= 0) & (u + w <= 1)
        t = torch.where(ok, t, torch.inf)
        tb, i = t.min(1)
        hit = torch.isfinite(tb)
        ub, wb = u.gather(1, i[:, None])[:, 0], w.gather(1, i[:, None])[:, 0]
        N = nn[i, 0] * (1 - ub - wb)[:, None] + nn[i, 1] * ub[:, None] + nn[i, 2] * wb[:, None]
        N = N / N.norm(dim=1, keepdim=True)
        best[0][a:b] = torch.where(hit[:, None], o[a:b] + tb[:, None].nan_to_num(posinf=0.0) * d[a:b], 0.0)
        best[1][a:b] = torch.where(hit[:, None], N, 0.0)
        best[2][a:b] = torch.where(hit[:, None], torch.stack([tb, ub, wb], 1),
                                   torch.tensor([torch.inf, 0.0, 0.0], dtype=torch.float64, device="cuda"))
    return {"point": best[0], "normal": best[1], "tuv": best[2], "ids": None}
