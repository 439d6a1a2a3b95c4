"""The segmented ray and shadow queues at the sizes where the dealing of
camera paths changes: films of one sample whose path counts lie around one
window (1024 paths), one round of windows over all segments (8192) and one
window more, against the oracle (counts exact, sums to the oracle's
rounding), with the smallest shading grid too; and the order of samples
within groups of 1024 pixels, and the rays that a wave begins with."""
import numpy as np
import pytest

import orc
from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from test_gpu_edges import _gpu_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(33, 31), (32, 32), (41, 25), (8191, 1), (128, 64), (2731, 3), (709, 13)],
                         ids=lambda s: str(s[0] * s[1]))
def test_paths_around_a_window(size):
    w, h = size
    desc = scenes.make_c0(width=w, height=h, spp=1, hdri_w=64, hdri_h=32)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
        upload_scene(integ, desc)
        osums = ocnt = None
        for shade in (0, 1):
            integ.setLaunch(shade_blocks_per_cu=shade)
            integ.resetIterationIndex()
            integ.render(1)
            sums, cnt = integ.readbackSums(), integ.counters()
            if ocnt is None:
                osums, ocnt = orc.Scene(desc, tables=_gpu_tables(integ, desc)).render("f32", samples=(0, 1))
            D = desc.max_depth + 1
            for k in ("rays", "hits", "shadow", "visible"):
                assert np.array_equal(cnt[k][:D], ocnt[k][:D]), (k, cnt[k][:D], ocnt[k][:D])
            assert cnt["rays"][1] == w * h
            # the oracle adds a path's radiances (at most 5 at depth 5) in
            # float32: at most 4 roundings of 2^-24 = 2.4e-7; the film in float64
            assert np.allclose(sums, osums, rtol=2.5e-7, atol=1e-30)


@pytest.mark.parametrize("size", [(1, 1), (33, 31), (32, 32), (41, 25), (683, 3), (61, 41)],
                         ids=lambda s: str(s[0] * s[1]))
def test_samples_around_a_pixel_group(size):
    """Several samples of films of less than one, one, just over one, just
    over two and several groups of pixels traced together, in batches of 2,
    2 and 1 samples and in one, in pixel rows and in tiles."""
    w, h = size
    desc = scenes.make_c0(width=w, height=h, spp=5, hdri_w=64, hdri_h=32)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
        upload_scene(integ, desc)
        osums, ocnt = orc.Scene(desc, tables=_gpu_tables(integ, desc)).render("f32", samples=(0, 5))
        D = desc.max_depth + 1
        for tile, spb in ((16, 0), (16, 2), (1, 0), (1, 2)):
            integ.setLaunch(tile=tile)
            integ.setParams(max_depth=desc.max_depth, rr_depth=desc.rr_depth, view=desc.view, samples_per_batch=spb)
            integ.resetIterationIndex()
            integ.render(5)
            sums, cnt = integ.readbackSums(), integ.counters()
            for k in ("rays", "hits", "shadow", "visible"):
                assert np.array_equal(cnt[k][:D], ocnt[k][:D]), (tile, spb, k)
            assert np.allclose(sums, osums, rtol=2.5e-7, atol=1e-30), (tile, spb)


@pytest.mark.parametrize("size", [(1, 1), (8, 8), (13, 5), (51, 5), (16, 16), (257, 1), (32, 16), (27, 19), (128, 64), (8193, 1)],
                         ids=lambda s: str(s[0] * s[1]))
def test_rays_spread_over_waves(size):
    """Segments whose ray counts lie around the limits below which a wave
    begins with 2 to 32 rays: with one traversal block per CU of 256, a
    segment has 128 waves and the limits are 64, 128, 256, 512 and 1024."""
    w, h = size
    desc = scenes.make_c0(width=w, height=h, spp=1, hdri_w=64, hdri_h=32)
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
        upload_scene(integ, desc)
        osums, ocnt = orc.Scene(desc, tables=_gpu_tables(integ, desc)).render("f32", samples=(0, 1))
        D = desc.max_depth + 1
        for blocks in (0, 1, 2):
            integ.setLaunch(trace_blocks_per_cu=blocks, shadow_blocks_per_cu=blocks)
            integ.resetIterationIndex()
            integ.render(1)
            sums, cnt = integ.readbackSums(), integ.counters()
            for k in ("rays", "hits", "shadow", "visible"):
                assert np.array_equal(cnt[k][:D], ocnt[k][:D]), (blocks, k)
            assert np.allclose(sums, osums, rtol=2.5e-7, atol=1e-30), blocks
