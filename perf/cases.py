"""The renderer's workloads as measurable cases, through its public entry points.

A case is one call sequence of a program that uses the renderer:

  frame      Integrator.render of one view, then the framebuffer on the host
  views      Integrator.renderViews of many views at once, then every view's image
  guided     a frame with the learned directional proposal (weights given)
  train      one Adam step of the learned proposal (Integrator.guideTrain)
  trace      closest hits or occlusion of rays in device memory
             (clhip_trace_rays_device)

Scenes are the repository's own seeded ones: "c0" (ground and 64 spheres under
sun and sky), "c1" (1080p terrain with 200 instanced spheres, 2.07 M triangles,
HDRI), "c3" (closed room lit through a window) and "textured" (texture-driven
materials).  A program uploads its scene once and then moves the camera, so
the contexts are kept per case and the seed decides the view: the camera's
position and the RNG lane (for the other kinds the rays, the samples and the
network's weights).
"""
from __future__ import annotations

import ctypes as C
import math
import random
from collections import OrderedDict
from dataclasses import replace

import numpy as np
import torch

from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from colvillea_amd import _capi as capi

SCENES = {"c0": scenes.make_c0, "c1": scenes.make_c1, "c3": scenes.make_c3, "textured": scenes.make_textured}
# eye, target, vertical field of view and how far the seed moves the eye
VIEWS = {"c0": ((0.0, 5.5, 11.0), (0.0, 0.5, 0.0), 45.0, 0.4), "c1": ((0.0, 7.0, 20.0), (0.0, 0.5, 0.0), 45.0, 0.5),
         "c3": ((0.0, 1.7, 4.6), (0.0, 1.0, -5.0), 65.0, 0.1),
         "textured": ((0.0, 3.2, 7.5), (0.0, 0.6, 0.0), 42.0, 0.2)}
# triangles and vertices stored, HDRI texels, and closest-hit and shadow rays
# of one camera path at the scene's own depth
STATS = {"c0": (1282, 646, 512 * 256, 2.2, 1.3), "c1": (1050626, 526850, 2048 * 1024, 1.8, 0.8),
         "c3": (185088, 94000, 2048 * 1024, 8.5, 6.5), "textured": (1282, 646, 256 * 128, 2.4, 1.6)}
MAX_CONTEXTS = 4

_scenes: dict = {}
_contexts: "OrderedDict" = OrderedDict()


def listed():
    return [
        # the smallest interactive call: a thumbnail refreshed at one sample
        # per pixel while a camera or a material is being dragged
        {"name": "preview_160x120_1spp", "kind": "frame", "scene": "c0", "width": 160, "height": 120, "spp": 1,
         "depth": 5, "rr": 3, "bvh": 4, "type": "path", "display": True},
        # a material preview: every texture slot and BSDF, odd film size
        {"name": "textured_321x241_4spp", "kind": "frame", "scene": "textured", "width": 321, "height": 241, "spp": 4,
         "depth": 6, "rr": 3, "bvh": 4, "type": "path", "display": True},
        # the small named configuration: 512x512, 16 spp, depth 5, roulette from 3
        {"name": "spheres_512_16spp", "kind": "frame", "scene": "c0", "width": 512, "height": 512, "spp": 16,
         "depth": 5, "rr": 3, "bvh": 4, "type": "path", "display": False},
        # the other integrator and the other tree width
        {"name": "direct_bvh8_961x541_8spp", "kind": "frame", "scene": "c1", "width": 961, "height": 541, "spp": 8,
         "depth": 2, "rr": 0, "bvh": 8, "type": "direct", "display": False},
        # a viewer's frame: render() adds one sample per pixel and the image is shown
        {"name": "viewer_1080p_1spp", "kind": "frame", "scene": "c1", "width": 1920, "height": 1080, "spp": 1,
         "depth": 8, "rr": 0, "bvh": 4, "type": "path", "display": True},
        # the headline: a 1080p still at 64 spp, depth 8
        {"name": "still_1080p_64spp", "kind": "frame", "scene": "c1", "width": 1920, "height": 1080, "spp": 64,
         "depth": 8, "rr": 0, "bvh": 4, "type": "path", "display": False},
        # long indoor paths: hardly any ray escapes before the depth limit
        {"name": "room_1080p_4spp", "kind": "frame", "scene": "c3", "width": 1920, "height": 1080, "spp": 4,
         "depth": 10, "rr": 0, "bvh": 4, "type": "path", "display": False},
        # a view server: 48 cameras of one scene in one batched call
        {"name": "views_48", "kind": "views", "scene": "c1", "set": 3, "count": 48, "side_min": 64, "side_max": 512,
         "spp_min": 4, "spp_max": 32, "depth_min": 3, "depth_max": 10},
        # the learned proposal in use: the room rendered with a given network
        {"name": "guided_room_960x540_4spp", "kind": "guided", "scene": "c3", "width": 960, "height": 540, "spp": 4,
         "depth": 10, "rr": 0, "fp8": False},
        # its training: one Adam step on 2^16 samples
        {"name": "train_65536", "kind": "train", "samples": 65536},
        # a baker's incoherent rays against the large scene, closest hits
        {"name": "trace_c1_1m", "kind": "trace", "scene": "c1", "rays": 1 << 20, "any": False, "bvh": 4},
        # visibility queries, a ragged and smaller batch
        {"name": "occlusion_c0_100003", "kind": "trace", "scene": "c0", "rays": 100003, "any": True, "bvh": 4},
    ]


def _log_int(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.55:
        scene = rng.choice(["c0", "c1", "c1", "c3", "textured"])
        w = _log_int(rng, 96, 1920)
        h = max(64, min(1080, int(round(w * rng.uniform(0.5, 1.0)))))
        budget = {"c0": 32e6, "c1": 64e6, "c3": 12e6, "textured": 32e6}[scene]  # camera paths of one pass
        spp = _log_int(rng, 1, max(1, min(64, budget / (w * h))))
        direct = rng.random() < 0.15
        return {"kind": "frame", "scene": scene, "width": w, "height": h, "spp": spp,
                "depth": 2 if direct else rng.randint(2, 12), "rr": rng.choice([0, 0, 3]),
                "bvh": 8 if rng.random() < 0.2 else 4, "type": "direct" if direct else "path",
                "display": rng.random() < 0.5}
    if u < 0.67:
        return {"kind": "views", "scene": "c1", "set": rng.randrange(1 << 16), "count": rng.randint(2, 60), "side_min": 64,
                "side_max": rng.randint(96, 512), "spp_min": 1, "spp_max": rng.randint(2, 32), "depth_min": 3,
                "depth_max": rng.randint(3, 10)}
    if u < 0.78:
        w = _log_int(rng, 96, 1280)
        h = max(64, int(round(w * rng.uniform(0.5, 0.8))))
        return {"kind": "guided", "scene": "c3", "width": w, "height": h,
                "spp": _log_int(rng, 1, max(1, min(16, 6e6 / (w * h)))), "depth": rng.randint(3, 10),
                "rr": rng.choice([0, 3]), "fp8": rng.random() < 0.3}
    if u < 0.88:
        return {"kind": "train", "samples": _log_int(rng, 8000, 300000)}
    return {"kind": "trace", "scene": rng.choice(["c0", "c1"]), "rays": _log_int(rng, 1000, 3e6),
            "any": rng.random() < 0.5, "bvh": 8 if rng.random() < 0.2 else 4}


# ------------------------------------------------------------------ contexts

def _scene(name):
    if name not in _scenes:
        _scenes[name] = SCENES[name]()
    return _scenes[name]


def _context(case, width, height):
    """The program's integrator with the scene uploaded, kept between states."""
    key = (case["kind"], case["scene"], width, height, case.get("bvh", 4), case.get("type", "path"))
    it = _contexts.pop(key, None)
    if it is None:
        while len(_contexts) >= MAX_CONTEXTS:
            _contexts.popitem(last=False)[1].close()
        kind = (IntegratorType.WavefrontDirectLighting if case.get("type") == "direct"
                else IntegratorType.WavefrontPathTracing)
        it = Integrator.createIntegrator(kind, width, height)
        it.setBVHWidth(case.get("bvh", 4))
        upload_scene(it, _scene(case["scene"]))
    _contexts[key] = it
    return it


def _camera(scene, width, height, rng):
    eye, at, fov, move = VIEWS[scene]
    eye = [e + rng.uniform(-move, move) for e in eye]
    return scenes.look_at(eye, at, (0, 1, 0), fov, width, height)


def _weights(rng):
    """A network of the shape training starts from: He-uniform layers, the
    output layer small and its unused columns zero; 256-64-64-64-64-64."""
    w = []
    for layer, n_in in enumerate((256, 64, 64, 64, 64)):
        m = rng.uniform(-1.0, 1.0, (n_in, 64)) * math.sqrt(6.0 / n_in)
        if layer == 4:
            m *= 0.5
            m[:, 40:] = 0.0
        w.append(m.reshape(-1))
    return np.concatenate(w).astype(np.float32)


def _samples(rng, n):
    """Training samples as the tracer gathers them: position in the unit box,
    unit normal and outgoing direction, a direction about the normal and a
    positive weight with a long tail that favours one side of the sky."""
    def unit(v):
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    nrm = unit(rng.standard_normal((n, 3)))
    wo = unit(rng.standard_normal((n, 3)) + nrm)
    wi = unit(rng.standard_normal((n, 3)) + 1.5 * nrm)
    wgt = np.exp(rng.standard_normal((n, 1)) + 3.0 * wi[:, 1:2])
    return np.concatenate([rng.uniform(0.0, 1.0, (n, 3)), nrm, wo, wi, wgt], 1).astype(np.float32)


def _rays(scene, n, any_hit, seed):
    """n rays (o, tmin, d, tmax): origins over the scene's floor area, all
    directions, a third of the rays aimed at the instances."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    half = (14.0, 7.0) if scene == "c1" else (4.0, 4.0)
    o = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float32)
    o = (o - torch.tensor([0.5, 0.0, 0.5], device="cuda")) * torch.tensor([2 * half[0], 3.0, 2 * half[1]], device="cuda")
    o[:, 1] += 0.2
    d = torch.randn(n, 3, generator=g, device="cuda", dtype=torch.float32)
    k = n // 3
    at = torch.from_numpy(np.ascontiguousarray(_scene(scene).instance_xform[1:, :, 3])).to("cuda")
    d[:k] = at[torch.randint(at.shape[0], (k,), generator=g, device="cuda")] - o[:k]
    d = d / d.norm(dim=1, keepdim=True)
    lo = torch.full((n, 1), 1e-3 if any_hit else 0.0, device="cuda")
    return torch.cat([o, lo, d, torch.full((n, 1), 3.4e38, device="cuda")], 1).contiguous()


# ------------------------------------------------------------------ the protocol

def prepare(case, seed):
    rng = random.Random(seed)
    kind = case["kind"]
    st = {"kind": kind}
    if kind in ("frame", "guided"):
        w, h = case["width"], case["height"]
        st.update(it=_context(case, w, h), camera=_camera(case["scene"], w, h, rng), lane=rng.randrange(4096),
                  spp=case["spp"], depth=case["depth"], rr=case["rr"], display=case.get("display", False))
        if kind == "guided":
            st["weights"] = _weights(np.random.default_rng(seed))
            st["fp8"] = case["fp8"]
    elif kind == "views":
        st["it"] = _context(case, 64, 64)
        # the films' sizes, samples and depths are the case's, the cameras the seed's
        films = scenes.make_c2_views(seed=case["set"], n_views=case["count"],
                                     side=(case["side_min"], case["side_max"]), spp=(case["spp_min"], case["spp_max"]),
                                     depth=(case["depth_min"], case["depth_max"]))
        cams = scenes.make_c2_views(seed=seed, n_views=case["count"])
        st["views"] = [replace(f, camera=c.camera, lane=rng.randrange(4096)) for f, c in zip(films, cams)]
    elif kind == "train":
        g = np.random.default_rng(seed)
        it = Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 16, 16)
        it.guideReset(1)
        it.setGuideWeights(_weights(g))
        st.update(it=it, samples=_samples(g, case["samples"]))
    else:
        n = case["rays"]
        st.update(it=_context(case, 16, 16), any=int(case["any"]), n=n, rays=_rays(case["scene"], n, case["any"], seed),
                  hit=torch.empty(n, 4, device="cuda"), prim=torch.empty(n, device="cuda", dtype=torch.int32))
        torch.cuda.synchronize()
    return st


def run(st):
    it = st["it"]
    kind = st["kind"]
    if kind in ("frame", "guided"):
        if kind == "guided":
            it.setGuideWeights(st["weights"])
            it.setGuide(True, precision=int(st["fp8"]))
        it.updateCamera(st["camera"])
        it.setParams(st["depth"], st["rr"], st["lane"])
        it.resetIterationIndex()
        it.render(st["spp"])
        return it.readbackFramebuffer() if st["display"] else it.readbackFramebufferLinear()
    if kind == "views":
        it.renderViews(st["views"])
        return [it.readbackView(i) for i in range(len(st["views"]))]
    if kind == "train":
        loss, grad = it.guideTrain(st["samples"], want_grad=True)
        return {"loss": loss, "grad": grad, "weights": it.guideWeights()}
    capi.check(capi.lib().clhip_trace_rays_device(it.ctx, st["rays"].data_ptr(), st["n"], st["any"],
                                                  st["hit"].data_ptr(), st["prim"].data_ptr()), it.ctx)
    # the hit record's fourth word is the instance index, not a number
    return {"occluded" if st["any"] else "t_b1_b2": st["hit"][:, :1] if st["any"] else st["hit"][:, :3],
            "instance": st["hit"].view(torch.int32)[:, 3], "prim": st["prim"]}


def work(case):
    """Bytes: scene records once (48 per triangle, 24 per vertex, 16 per
    texel), inputs once, outputs once.  Flops: per ray one descent of a
    4-wide tree (4 boxes of 12 per level) and a triangle test, per closest
    hit about 400 of shading; the network's products where it runs."""
    kind = case["kind"]
    if kind == "train":
        n = case["samples"]
        return {"bytes": 52 * n + 7 * 4 * 32768, "flops": 163840 * n}
    tris, verts, texels, cr, sr = STATS[case["scene"]]
    scene = 48 * tris + 24 * verts
    per_ray = 48 * math.ceil(math.log(tris, 4)) + 60
    if kind == "trace":
        return {"bytes": scene + 52 * case["rays"], "flops": per_ray * case["rays"]}
    if kind == "views":
        # the mean of a log-uniform side's square, uniform spp
        lo, hi = case["side_min"], case["side_max"]
        area = (hi * hi - lo * lo) / (2.0 * math.log(hi / lo)) if hi > lo else lo * lo
        pixels = case["count"] * area
        paths = pixels * 0.5 * (case["spp_min"] + case["spp_max"])
        depth = 0.5 * (case["depth_min"] + case["depth_max"])
    else:
        pixels = case["width"] * case["height"]
        paths = pixels * case["spp"]
        depth = case["depth"]
    closest, shadow = min(cr, depth), min(sr, depth - 1.0)
    flops = paths * ((closest + shadow) * per_ray + closest * 400.0)
    if kind == "guided":
        flops += paths * (closest - 1.0) * 65536.0
    return {"bytes": scene + 16 * texels + 16 * pixels, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "train":
        # bfloat16 operands: the gradient's rounding; Adam turns it into
        # steps of the learning rate where a gradient is near zero
        return {"rel": 1e-2, "max": 0.5}
    if kind == "trace":
        # float32 hits; whole values may differ where a ray meets an edge
        # shared by two triangles at equal distance
        return {"rel": 1e-6, "max": 1e-4, "differ": 1e-5}
    # the film is a float64 sum of float32 radiances in any order, rounded to
    # float32 once (and encoded by powf for display): the last bit may differ
    return {"rel": 1e-6, "max": 1e-5}


# ------------------------------------------------------------------ 64-bit values

def _exact_trace(case, seed):
    """Closest hits (t, b1, b2) or occlusion against every triangle of the
    ground-and-spheres scene in float64: per instance, the ray's moment
    against every edge gives the signed volumes of the triangle test."""
    desc = _scene(case["scene"])
    rays = _rays(case["scene"], case["rays"], case["any"], seed).double()
    o, d, tmin = rays[:, :3], rays[:, 4:7], rays[:, 3]
    n = rays.shape[0]
    best = torch.full((n, 3), 0.0, device="cuda", dtype=torch.float64)
    best[:, 0] = math.inf
    for mesh_i, xf in zip(desc.instance_mesh, desc.instance_xform):
        mesh = desc.meshes[mesh_i]
        m = torch.from_numpy(xf.astype(np.float64)).cuda()
        v = torch.from_numpy(mesh.vertices.astype(np.float64)).cuda() @ m[:, :3].T + m[:, 3]
        tri = v[torch.from_numpy(mesh.triangles.astype(np.int64)).cuda()]  # (m, 3, 3)
        c = v.mean(0)
        r = (v - c).norm(dim=1).max() * 1.0001
        # rays that can meet the mesh's bounding sphere
        b = ((c - o) * d).sum(1)
        near = torch.nonzero(((c - o) - b[:, None] * d).norm(dim=1) <= r).squeeze(1)
        e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
        nrm = torch.linalg.cross(e1, e2)
        for s in range(0, near.numel(), 16384):
            i = near[s:s + 16384]
            oi, di = o[i], d[i]
            mom = torch.linalg.cross(oi, di)  # side product of the ray with an edge p -> q: d.(p x q) + mom.(q - p)
            vol = []
            for p, q in ((1, 2), (2, 0), (0, 1)):
                pq = torch.linalg.cross(tri[:, p], tri[:, q])
                vol.append(di @ pq.T + mom @ (tri[:, q] - tri[:, p]).T)
            same = ((vol[0] >= 0) & (vol[1] >= 0) & (vol[2] >= 0)) | ((vol[0] <= 0) & (vol[1] <= 0) & (vol[2] <= 0))
            det = vol[0] + vol[1] + vol[2]
            t = ((tri[:, 0] * nrm).sum(1)[None, :] - oi @ nrm.T) / (di @ nrm.T)
            t = torch.where(same & (det != 0) & (t >= tmin[i][:, None]), t, math.inf)
            tb, j = t.min(1)
            k = torch.arange(i.numel(), device="cuda")
            cand = torch.stack([tb, vol[1][k, j] / det[k, j], vol[2][k, j] / det[k, j]], 1)
            best[i] = torch.where((tb < best[i, 0])[:, None], cand, best[i])
    hit = torch.isfinite(best[:, 0])
    if case["any"]:
        return {"occluded": hit.double()[:, None], "instance": None, "prim": None}
    best[~hit] = torch.tensor([-1.0, 0.0, 0.0], device="cuda", dtype=torch.float64)
    return {"t_b1_b2": best, "instance": None, "prim": None}


def _exact_train(case, seed):
    """Loss, gradient and Adam's first step of the mixture's weighted negative
    log-likelihood, by float64 autograd."""
    g = np.random.default_rng(seed)
    p = torch.from_numpy(_weights(g).astype(np.float64)).cuda().requires_grad_()
    s = torch.from_numpy(_samples(g, case["samples"]).astype(np.float64)).cuda()
    q, wi, wgt = s[:, :9], s[:, 9:12], s[:, 12]
    feat = []
    for dim in range(9):
        for f in range(12):
            a = math.pi * 2.0 ** f * q[:, dim]
            feat += [torch.sin(a), torch.cos(a)]
    x = torch.stack(feat + [q[:, k] for k in range(9)] + [torch.ones_like(wgt)], 1)
    x = torch.cat([x, torch.zeros(x.shape[0], 256 - x.shape[1], device="cuda", dtype=torch.float64)], 1)
    off = 0
    for layer, n_in in enumerate((256, 64, 64, 64, 64)):
        x = x @ p[off:off + n_in * 64].reshape(n_in, 64)
        off += n_in * 64
        if layer < 4:
            x = torch.relu(x)
    out = x[:, :40].reshape(-1, 8, 5)
    kappa = torch.exp(out[..., 4].clamp(-4.0, 8.0))
    mu = out[..., 1:4] / out[..., 1:4].norm(dim=2, keepdim=True)
    logp = (torch.log_softmax(out[..., 0], 1) + torch.log(kappa) - math.log(2.0 * math.pi)
            - torch.log(-torch.expm1(-2.0 * kappa)) + kappa * ((mu * wi[:, None, :]).sum(2) - 1.0))
    loss = -(wgt / wgt.sum() * torch.logsumexp(logp, 1)).sum()
    loss.backward()
    grad = p.grad
    # Adam's bias-corrected first step: m = g, v = g^2
    step = 1e-3 * grad / (grad.abs() + 1e-8)
    return {"loss": loss.detach(), "grad": grad, "weights": (p - step).detach()}


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "trace" and case["scene"] == "c0" and case["rays"] <= 1 << 18:
        return _exact_trace(case, seed)
    # c1 has 2.07 M triangles: every triangle against every ray takes too
    # long.  And an image is not a 64-bit computation's rounded value: a path
    # takes its turns (lobes, hits at grazing angles, texels) by comparing
    # 32-bit numbers, so a 64-bit renderer walks other paths.
    return None
