"""The renderer's performance cases: what a program that uses rayna_amd has it do, through its public entry points.

A case names a scene of rayna_amd.presets, a frame size, samples per pixel and how the frame is asked for:
  render      Renderer.render after clear_accumulation: the first frame of a scene, the float image on the host
  preview     the interactive loop: the camera is set again, then `frames` accumulating frames as 8-bit RGBA
  step        one step of inverse rendering: ColourRenderer's forward frame and the gradient of an L2 image loss
  batch       BatchRenderer.render of `requests` requests of mixed scenes, sizes and sample counts
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rayna_amd import Renderer, presets
from rayna_amd.batch import BatchRenderer
from rayna_amd.diff import ColourRenderer
from rayna_amd.scene import (Camera, DielectricMaterial, LambertianMaterial, MetalMaterial, RenderMode, RenderOpts)

SCENES = ("spheres", "cornell", "rttnw", "mesh", "sdf", "textured", "mixed")


def listed():
    return [
        # the smallest call: a thumbnail, where launches and latency are all there is
        dict(name="spheres thumbnail", call="render", scene="spheres", width=64, height=36, samples=2, depth=6),
        # the book's demo frame at the preset's size
        dict(name="spheres frame", call="render", scene="spheres", width=400, height=225, samples=32, depth=10),
        # parallelograms and rotated boxes under one light, closed room: every path runs to the depth limit
        dict(name="cornell frame", call="render", scene="cornell", width=600, height=600, samples=64, depth=8),
        # a scattering medium, an instanced cloud of balls and a noise texture
        dict(name="rttnw frame", call="render", scene="rttnw", width=600, height=600, samples=32, depth=10),
        # a user moving the camera over a mesh: four one-sample frames at a window's odd size, 8-bit output
        dict(name="mesh preview", call="preview", scene="mesh", subdiv=6, width=641, height=359, samples=1, depth=5,
             frames=4),
        # the benchmark frame: 1.3 million triangles at 1080p
        dict(name="mesh 1080p", call="render", scene="mesh", subdiv=8, width=1920, height=1080, samples=64, depth=8),
        # a small frame of the ray-marched scene, as a request of a serving batch has it
        dict(name="sdf small", call="render", scene="sdf", width=161, height=91, samples=9, depth=12),
        # the ray-marched scene at the preset's size: the longest frame
        dict(name="sdf 720p", call="render", scene="sdf", width=1280, height=720, samples=128, depth=12),
        # every texture kind, an image sky, odd sizes, a sample count that is not a square
        dict(name="textured odd", call="render", scene="textured", width=333, height=217, samples=10, depth=6),
        # a debug view (outward normals) over every primitive kind
        dict(name="normals view", call="render", scene="mixed", width=960, height=540, samples=4, depth=6,
             mode="OutwardNormal"),
        # forward and backward of one inverse-rendering step at the workload's size
        dict(name="inverse step", call="step", width=256, height=256, samples=16, depth=10),
        # a serving batch: requests of three scenes, 128x128 to 640x360, 1 to 64 samples
        dict(name="batch of 16", call="batch", requests=16, subdiv=6, width=640, height=360, samples=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(("render", "render", "render", "render", "preview", "step", "batch"))
    if call == "step":
        side = _log_int(rng, 32, 256)
        return dict(call=call, width=side, height=rng.randint(max(16, side // 2), side), samples=_log_int(rng, 1, 16),
                    depth=rng.randint(3, 10))
    if call == "batch":
        return dict(call=call, requests=rng.randint(2, 16), subdiv=rng.randint(3, 6), width=rng.randint(160, 640),
                    height=rng.randint(130, 360), samples=_log_int(rng, 2, 64))
    if call == "preview":
        return dict(call=call, scene=rng.choice(("mesh", "spheres", "cornell")), subdiv=rng.randint(3, 7),
                    width=_log_int(rng, 160, 1280), height=_log_int(rng, 90, 720), samples=rng.randint(1, 4),
                    depth=rng.randint(3, 8), frames=rng.randint(1, 6))
    scene = rng.choice(SCENES)
    case = dict(call=call, scene=scene, width=_log_int(rng, 48, 1280), height=_log_int(rng, 32, 720),
                samples=_log_int(rng, 1, 64), depth=rng.randint(3, 10))
    if scene == "mesh":
        case["subdiv"] = rng.randint(3, 8)
    if rng.random() < 0.1:
        case["mode"] = rng.choice(("RayNormal", "OutwardNormal", "Scatter", "FrontFace", "Distance", "Uv", "Side"))
    return case


def _scene(case, seed):
    """(scene, camera, options) of a case: the preset with the case's frame, everything random in it from `seed`."""
    size = dict(width=case["width"], height=case["height"], samples=case["samples"], ray_depth=case["depth"])
    if case["scene"] == "mesh":
        scene, cam, opts = presets.triangle_mesh(seed=seed, subdiv=case["subdiv"], **size)
    else:
        make = {"spheres": presets.random_spheres, "cornell": presets.cornell, "rttnw": presets.rttnw,
                "sdf": presets.sdf_volume, "textured": presets.textured, "mixed": presets.mixed_primitives}
        scene, cam, opts = make[case["scene"]](seed=seed, **size)
    mode = RenderMode[case.get("mode", "PBR")]
    return scene, cam, RenderOpts(opts.width, opts.height, opts.samples, opts.ray_depth, mode=int(mode), seed=seed)


def prepare(case, seed):
    if case["call"] == "step":
        scene, cam, opts, hidden = presets.inverse_spheres(seed=seed, width=case["width"], height=case["height"],
                                                           samples=case["samples"], ray_depth=case["depth"])
        rng = np.random.default_rng(seed)
        colours = scene.colours()
        colours[hidden] = rng.uniform(0.1, 0.9, (len(hidden), 3))
        target = rng.uniform(0.0, 1.0, (case["height"], case["width"], 3)).astype(np.float32)
        return dict(call="step", f=ColourRenderer(scene, cam, opts), target=torch.from_numpy(target),
                    colours=torch.from_numpy(colours).requires_grad_(True), seed=opts.seed)
    if case["call"] == "batch":
        # the preset's draw of scenes, sizes and sample counts; every request with a random stream of its own
        scenes, requests = presets.batch_requests(n=case["requests"], mesh_subdiv=case["subdiv"], max_w=case["width"],
                                                  max_h=case["height"], max_spp=case["samples"])
        for k, q in enumerate(requests):
            q.opts.seed = 1000 * seed + k
        batch = BatchRenderer(scenes)
        batch.set_tuning(schedule="interleaved")
        return dict(call="batch", batch=batch, requests=requests)
    scene, cam, opts = _scene(case, seed)
    return dict(call=case["call"], renderer=Renderer.new_from(scene, cam, opts), camera=cam,
                frames=case.get("frames", 1))


def run(state):
    if state["call"] == "step":
        colours = state["colours"]
        colours.grad = None
        img = state["f"](colours, seed=state["seed"])
        loss = ((img - state["target"]) ** 2).mean()
        loss.backward()
        return {"image": img.detach(), "grad": colours.grad}
    if state["call"] == "batch":
        return state["batch"].render(state["requests"])[0]
    r = state["renderer"]
    if state["call"] == "preview":
        r.set_camera(state["camera"])
        for _ in range(state["frames"]):
            out = r.render_srgb8()
        return out.img
    r.clear_accumulation()
    return r.render(layout="rowmajor").img


def work(case):
    """Bytes: the scene's records read once and the image written once.  Floating-point operations: per sample its
    camera ray and two closest-hit queries with their shading, per query a binary tree's levels (two boxes each), a
    few primitive tests, or a ray march of a few dozen distance estimates."""
    if case["call"] == "batch":
        prims, bytes_each, march = 20 * 4 ** case["subdiv"] + 500, 96, 1.0 / 3.0
        pixels = case["requests"] * math.sqrt(128.0 * 128.0 * case["width"] * case["height"])
        samples = pixels * (case["samples"] + 1) / 2
    else:
        scene = case.get("scene", "spheres")
        prims = {"spheres": 480, "cornell": 8, "rttnw": 1410, "sdf": 18, "textured": 7, "mixed": 60,
                 "mesh": 20 * 4 ** case.get("subdiv", 0) + 10}[scene]
        bytes_each, march = 96, scene == "sdf"
        pixels = case["width"] * case["height"]
        samples = pixels * case["samples"] * case.get("frames", 1)
    queries = samples * (1 if case.get("mode", "PBR") != "PBR" else 4 if case["call"] == "step" else 2)
    per_query = 24 * 2 * math.ceil(math.log2(prims)) + 4 * 50 + 200 + 30 * 500 * march
    out = pixels * (4 if case["call"] == "preview" else 12)
    return {"bytes": prims * bytes_each + out, "flops": queries * per_query}


# ---------------------------------------------------------------------------- the sphere scenes in 64 bits


def _philox(c, key):
    """Philox4x32-10 (Salmon et al., SC 2011) of four int64 tensors holding 32-bit words."""
    m32 = 0xFFFFFFFF
    k0, k1 = key
    c0, c1, c2, c3 = c
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & m32) ^ c1 ^ k0, p1 & m32, ((p0 >> 32) & m32) ^ c3 ^ k1, p0 & m32
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    return torch.stack([c0, c1, c2, c3], 1)


def _uniforms(pixel, sample, bounce, slot, seed):
    word = _philox((pixel, sample, torch.full_like(pixel, bounce), torch.full_like(pixel, slot)),
                   (seed & 0xFFFFFFFF, seed >> 32))
    return (word >> 8).double() * 2.0 ** -24


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True)


def _on_sphere(u, v):
    q = 2.0 * torch.sqrt(v * (1.0 - v))
    return torch.stack([torch.cos(2 * math.pi * u) * q, torch.sin(2 * math.pi * u) * q, 1.0 - 2.0 * v], 1)


def _camera_rays(cam: Camera, opts: RenderOpts, pixel, sample):
    """Stratified jitter in a grid of isqrt(samples) squared cells, a thin lens of the camera's defocus angle."""
    f8 = dict(dtype=torch.float64, device=pixel.device)
    u = _uniforms(pixel, sample, 0, 0, opts.seed)
    x, y = (pixel % opts.width).double() + u[:, 0] - 0.5, (pixel // opts.width).double() + u[:, 1] - 0.5
    s = math.isqrt(opts.samples)
    cell = sample < s * s
    cx = torch.where(cell, (pixel % opts.width) + ((u[:, 0] - 0.5) + (sample % s)) / s, x)
    cy = torch.where(cell, (pixel // opts.width) + ((u[:, 1] - 0.5) + (sample // s)) / s, y)
    w = -_unit(torch.tensor(cam.fwd, **f8))
    right = _unit(torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0], **f8), w))
    up = torch.linalg.cross(w, right)
    pos = torch.tensor(cam.pos, **f8)
    size = 2.0 * math.tan(math.radians(cam.v_fov) / 2.0) * cam.focus_dist
    lens = cam.focus_dist * math.tan(math.radians(cam.defocus_angle) / 2.0)
    at = (pos - w * cam.focus_dist + right * (size * (cx - opts.width / 2.0) / opts.height)[:, None]
          - up * (size * (cy - opts.height / 2.0) / opts.height)[:, None])
    r, a = lens * torch.sqrt(u[:, 2]), 2 * math.pi * u[:, 3]
    org = pos + right * (r * torch.cos(a))[:, None] + up * (r * torch.sin(a))[:, None]
    return org, _unit(at - org)


def _closest(centre, radius, org, d):
    oc = org[:, None] - centre[None]
    b, c = (oc * d[:, None]).sum(-1), (oc * oc).sum(-1) - radius ** 2
    root = torch.sqrt(b * b - c)  # NaN on a miss, which no comparison keeps
    near, far = -b - root, -b + root
    inf = torch.full_like(near, math.inf)
    return torch.where(near >= 1e-3, near, torch.where(far >= 1e-3, far, inf)).min(1)


def _paths(scene, cam, opts, pixel, sample):
    """The radiance of each sample: spheres of diffuse, metal and glass under the gradient sky, every random number
    from the counter (pixel, sample, bounce, 1)."""
    f8 = dict(dtype=torch.float64, device=pixel.device)
    centre = torch.tensor(np.array([o.mesh.pos for o in scene.objects]), **f8)
    radius = torch.tensor([float(o.mesh.radius) for o in scene.objects], **f8)
    mats = [o.material for o in scene.objects]
    kind = torch.tensor([(LambertianMaterial, MetalMaterial, DielectricMaterial).index(type(m)) for m in mats],
                        device=pixel.device)
    albedo = torch.tensor(np.array([m.albedo for m in mats]), **f8)
    fuzz = torch.tensor([getattr(m, "fuzz", 0.0) for m in mats], **f8)
    out = torch.zeros((len(pixel), 3), **f8)
    live = torch.arange(len(pixel), device=pixel.device)
    org, d = _camera_rays(cam, opts, pixel, sample)
    weight = torch.ones_like(org)
    for bounce in range(opts.ray_depth + 1):
        parts = [_closest(centre, radius, o, e) for o, e in zip(org.split(32768), d.split(32768))]
        t, obj = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
        miss = torch.isinf(t)
        a = 0.5 * d[miss, 1:2] + 0.5
        out[live[miss]] += weight[miss] * (1.0 + torch.tensor([-0.5, -0.3, 0.0], **f8) * a)
        if bounce == opts.ray_depth:
            break
        live, org, d, weight, t, obj = (v[~miss] for v in (live, org, d, weight, t, obj))
        pos = org + d * t[:, None]
        n = (pos - centre[obj]) / radius[obj][:, None]
        front = ~((d * n).sum(-1) > 0)
        n = torch.where(front[:, None], n, -n)
        u = _uniforms(pixel[live], sample[live], bounce, 1, opts.seed)
        ball = _on_sphere(u[:, 0], u[:, 1])
        diffuse = _unit(n + ball * u[:, 2:3] ** (1.0 / 3.0))
        mirror = d - n * (2.0 * (d * n).sum(-1, keepdim=True))
        metal = mirror + ball * fuzz[obj][:, None]
        absorbed = (kind[obj] == 1) & ~((metal * n).sum(-1) > 0)
        ratio = torch.where(front, 1.0 / 1.5, 1.5)  # every glass sphere of these scenes has index 1.5
        cos = (-(d * n).sum(-1)).clamp(max=1.0)
        r0 = ((1.0 - ratio) / (1.0 + ratio)) ** 2
        bends = ~((ratio * torch.sqrt(1.0 - cos * cos) > 1.0) | (r0 + (1.0 - r0) * (1.0 - cos) ** 5 > u[:, 0]))
        perp = (d + n * cos[:, None]) * ratio[:, None]
        through = perp - n * torch.sqrt((1.0 - (perp * perp).sum(-1, keepdim=True)).abs())
        glass = torch.where(bends[:, None], through, mirror)
        k = kind[obj][:, None]
        d = _unit(torch.where(k == 0, diffuse, torch.where(k == 1, metal, glass)))
        weight = torch.where((k == 2) & front[:, None], weight, weight * albedo[obj])
        live, org, d, weight = (v[~absorbed] for v in (live, pos, d, weight))
    return out


def exact(case, seed):
    """The sphere scenes' frames, every sphere tested by every ray in 64 bits.  The other scenes' meshes, marches and
    media have no such short statement."""
    paths = case["width"] * case["height"] * case["samples"]
    if case["call"] != "render" or case["scene"] != "spheres" or case.get("mode", "PBR") != "PBR" or paths > 1 << 22:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if dev == "cpu" and paths > 1 << 15:
        return None
    scene, cam, opts = _scene(case, seed)
    slot = torch.arange(paths, device=dev)
    colour = _paths(scene, cam, opts, slot // opts.samples, slot % opts.samples)
    return colour.reshape(opts.height, opts.width, opts.samples, 3).mean(2).cpu().numpy()
