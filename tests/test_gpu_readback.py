"""Film readback through pinned staging, at sizes around its 1 MiB pieces,
the two pieces from which several threads copy, and its 32 MiB of slots: the
linear film equals the float64 sums over the samples, and both equal the film
of a batched render of the same view.  Twice in a row with other samples, so
that a stale piece shows.  Training samples take the same way up: one Adam
step on a large batch equals the step on the same samples in a fresh context,
and the loss of the rows at the edges of the copy's parts is the oracle's."""
import ctypes as C

import numpy as np
import pytest

import guide_ref as G
from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from colvillea_amd import _capi as capi
from colvillea_amd.integrator import View
from test_zz_no_alloc import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(3, 2), (256, 256), (257, 256), (512, 256), (513, 256), (1447, 1451)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
def test_film_readback(size):
    w, h = size
    desc = scenes.make_c0(width=w, height=h, spp=1, hdri_w=64, hdri_h=32)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
        upload_scene(integ, desc)
        for lane in (0, 7):
            integ.setParams(2, 0, lane)
            integ.resetIterationIndex()
            integ.render(2)
            sums = integ.readbackSums()
            img = integ.readbackFramebufferLinear()
            integ.renderViews([View(w, h, 2, 2, desc.camera, 0, lane)])
            # one NEE term and the escape per path: the sums are exact in any order up to float64 rounding
            assert np.allclose(integ.readbackViewSums(0), sums, rtol=1e-14, atol=0)
            assert np.array_equal(img[..., :3], (sums * 0.5).astype(np.float32))
            assert np.all(img[..., 3] == 1.0)
            assert np.allclose(integ.readbackView(0), img, rtol=1e-6, atol=0)


def test_readback_into_pinned_memory():
    w, h = 512, 300  # 2.3 MiB
    desc = scenes.make_c0(width=w, height=h, spp=1, hdri_w=64, hdri_h=32)
    hip = DeviceArray.hip()
    own = C.c_void_p()
    assert hip.hipHostMalloc(C.byref(own), C.c_size_t(16 * w * h), 0) == 0
    try:
        out = np.ctypeslib.as_array(C.cast(own, C.POINTER(C.c_float)), (h, w, 4))
        out[:] = 7.0
        with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
            upload_scene(integ, desc)
            integ.render(1)
            capi.check(capi.lib().clhip_readback(integ.ctx, C.cast(own, C.POINTER(C.c_float)), out.nbytes), integ.ctx)
            assert np.array_equal(out, integ.readbackFramebufferLinear())
    finally:
        hip.hipHostFree(own)


@pytest.mark.parametrize("n", [1, 20165, 20166, 40329, 40330, 60000, 80661, 700001])
def test_training_samples_upload(n):
    rng = np.random.default_rng(n)
    unit = lambda v: v / np.linalg.norm(v, axis=1, keepdims=True)
    s = np.concatenate([rng.uniform(0, 1, (n, 3)), unit(rng.normal(size=(n, 3))), unit(rng.normal(size=(n, 3))),
                        unit(rng.normal(size=(n, 3))), rng.uniform(0.1, 2.0, (n, 1))], 1).astype(np.float32)
    out = []
    for first in (False, True):
        with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8) as integ:
            integ.guideReset(3)
            if first:  # leave other samples in the staging, then start over
                integ.guideTrain(s[::-1].copy())
                integ.guideReset(3)
            loss, g = integ.guideTrain(s, want_grad=True)
            assert integ.guideStats()["last_count"] == n
            out.append((loss, g, integ.guideWeights()))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])
    assert np.any(out[0][1])

    # only the rows at the ends and at the first edges of 2 MiB parts carry
    # weight: a stale piece would bring in thousands of weighted rows
    cut = np.arange(0, 52 * n, 2 << 20)[:4] // 52
    rows = np.unique(np.clip(np.concatenate([cut - 1, cut, cut + 1, [n - 1]]), 0, n - 1))
    w = s[rows, 12].astype(np.float64)
    t = s.copy()
    t[:, 12] = 0.0
    t[rows, 12] = s[rows, 12]
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 8, 8) as integ:
        integ.guideReset(3)
        integ.guideTrain(s[::-1].copy())
        integ.guideReset(3)
        Ws = G.split_params(integ.guideWeights().astype(np.float64))
        Ws[4][:, :40] *= 10.0  # densities that differ from sample to sample
        p = G.join_params(Ws).astype(np.float32)
        integ.setGuideWeights(p)
        loss, _ = integ.guideTrain(t)
    out, _ = G.forward(G.split_params(p.astype(np.float64)), G.encode(t[rows, :9].astype(np.float64)), bf=True)
    each = -np.log(G.mix_pdf(out, t[rows, 9:12].astype(np.float64)))
    ref = (w * each).sum() / w.sum()
    # 1e-3: the bound of the gradient test for the same bfloat16 network; one
    # wrong row among these shifts the loss by its share of |each - ref|
    assert abs(loss - ref) <= 1e-3 * abs(ref), (loss, ref)
    assert n == 1 or (w / w.sum() * np.abs(each - ref)).max() > 1e-3 * abs(ref)
