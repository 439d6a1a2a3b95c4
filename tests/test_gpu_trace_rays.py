"""Given-ray tracing on a persistent grid: a ray's result does not depend on
its place or on how many rays the call holds -- one ray, the sizes around a
wave and a block, and more rays than the grid has lanes -- for closest hit
and any hit, on both tree widths, with tmin and tmax of each ray's own.
(The hits themselves are checked against brute force in test_gpu_parity.)"""
import ctypes as C

import numpy as np
import pytest

from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from colvillea_amd import _capi as capi
from colvillea_amd.integrator import TriangleMesh
from test_zz_no_alloc import rays, trace_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
def test_results_do_not_depend_on_the_batch(width):
    desc = scenes.make_c0(width=8, height=8, spp=1, hdri_w=32, hdri_h=16)
    n = 700001  # the largest grid has 327680 lanes
    r = rays(desc, n, 11, 0.0)
    rng = np.random.default_rng(12)
    r[:, 3] = rng.choice([0.0, 1e-3, 2.0], n)
    r[:, 7] = rng.choice([1.0, 5.0, 3.4e38], n)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8) as integ:
        integ.setBVHWidth(width)
        upload_scene(integ, desc)
        for any_hit in (False, True):
            hit, prim = trace_device(integ, r, any_hit)
            assert 0.05 < (hit[:, 0] > 0).mean() < 0.95
            at = 0
            for m in (1, 63, 64, 65, 255, 257, 30011):
                h, p = trace_device(integ, r[at:at + m], any_hit)
                assert np.array_equal(h.view(np.uint32), hit[at:at + m].view(np.uint32)), m
                assert np.array_equal(p, prim[at:at + m]), m
                at += m
            occ = np.zeros(n, np.uint8)
            if any_hit:
                capi.check(capi.lib().clhip_occlusion_batch(integ.ctx, capi.fptr(r), n,
                                                            occ.ctypes.data_as(C.POINTER(C.c_uint8))), integ.ctx)
                assert np.array_equal(occ != 0, hit[:, 0] != 0)


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
@pytest.mark.parametrize("far", [1e3, 1e12, 1e19, 1e21])
def test_a_near_triangle_beside_a_far_one(width, far):
    """Both lie in one node, whose extent is up to 1e21: rays along the axes
    (reciprocals up to 1e20) through the near one still hit it."""
    near = np.array([[-1, -1, -5], [3, -1, -5], [-1, 3, -5]], np.float32)
    v = np.concatenate([near, near + np.float32([-far, 0, 0]), near + np.float32([0, -far, 0])]).astype(np.float32)
    mesh = TriangleMesh(v, np.arange(9, dtype=np.uint32).reshape(3, 3))
    r = np.array([[0.25 * i, 0.25 * j, 0, 0, 0, 0, -1, 3e38] for i in range(3) for j in range(3)], np.float32)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8) as integ:
        integ.setBVHWidth(width)
        integ.buildBLAS([mesh])
        integ.buildTLAS([mesh], [0])
        for any_hit in (False, True):
            hit, prim = trace_device(integ, r, any_hit)
            assert np.all(hit[:, 0] == (1.0 if any_hit else 5.0)) and np.all(prim == 0), (hit, prim)


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
def test_rays_without_a_place_or_direction_miss(width):
    """NaN in a ray lets it into every box, also the empty slots' (they hold
    no reference): it misses, and the rays beside it keep their hits."""
    ball = scenes.icosphere(1)
    xf = np.stack([scenes.IDENTITY, scenes.translate_scale((2.5, 0.0, 0.0), 0.7), scenes.translate_scale((0.0, 2.5, 0.0), 0.4)])
    rng = np.random.default_rng(2)
    n = 192
    o = rng.uniform(-4.0, 4.0, (n, 3))
    d = rng.uniform(-1.0, 1.0, (n, 3)) + [[0.8, 0.8, 0.0]] - o
    good = np.concatenate([o, np.zeros((n, 1)), d / np.linalg.norm(d, axis=1, keepdims=True), np.full((n, 1), 3e38)],
                          1).astype(np.float32)
    bad = good.copy()
    at = np.arange(0, n, 3)
    for i, k in enumerate(at):
        bad[k, [[0], [0, 1, 2], [4], [4, 5, 6], [0, 1, 2, 4, 5, 6]][i % 5]] = np.nan if i % 2 else np.inf
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8) as integ:
        integ.setBVHWidth(width)
        integ.buildBLAS([ball])
        integ.buildTLAS([ball] * 3, [0, 1, 2], xf.astype(np.float32))
        for any_hit in (False, True):
            ref, ref_prim = trace_device(integ, good, any_hit)
            hit, prim = trace_device(integ, bad, any_hit)
            rest = np.setdiff1d(np.arange(n), at)
            assert np.array_equal(hit[rest].view(np.uint32), ref[rest].view(np.uint32)) and (ref[rest, 0] > 0).sum() > 20
            assert np.array_equal(prim[rest], ref_prim[rest])
            assert np.all(hit[at, 0] == (0.0 if any_hit else -1.0)), hit[at, 0]
