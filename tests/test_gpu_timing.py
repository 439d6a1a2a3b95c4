"""A timed render issues closest hit and any hit as launches of their own at
every depth, an untimed one shares a launch between a depth's shadow rays and
the next depth's closest hits: both trace the same rays through the same
nodes and triangles, into the same film, for one view and for many (whose
camera rays read their origins), for grids whose lanes refill and for small
films, and for a guided render that records its paths."""
import numpy as np
import pytest

from colvillea_amd import Integrator, IntegratorType, scenes, upload_scene
from colvillea_amd.integrator import View

pytestmark = pytest.mark.gpu

COUNTS = ("rays", "hits", "shadow", "visible")
WORK = ("trace_nodes", "trace_tris", "shadow_nodes", "shadow_tris")


def _same(a, b):
    for k in COUNTS:
        assert np.array_equal(a[k], b[k]), (k, a[k], b[k])
    for k in WORK:
        assert a[k] == b[k] and a[k] > 0, (k, a[k], b[k])


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
@pytest.mark.parametrize("size,blocks", [((24, 17), 0), ((320, 240), 0), ((320, 240), 1)], ids=["small", "large", "refill"])
def test_timed_render_equals_untimed(width, size, blocks):
    w, h = size
    desc = scenes.make_textured(width=w, height=h, spp=4, hdri_w=64, hdri_h=32)
    views = [View(w, h, 2, 5, desc.camera, 0, 1), View(33, 21, 3, 4, desc.camera, 2, 2)]
    out = []
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, w, h) as integ:
        integ.setBVHWidth(width)
        upload_scene(integ, desc)
        # 65536 lanes serve 307200 camera rays with one block per CU
        integ.setLaunch(trace_blocks_per_cu=blocks, shadow_blocks_per_cu=blocks)
        for timed in (True, False):
            integ.setTiming(timed)
            integ.resetIterationIndex()
            integ.render(4)
            film, cnt = integ.readbackSums(), integ.counters()
            assert (cnt["trace_ms"] > 0 and cnt["shadow_ms"] > 0) == timed
            integ.renderViews(views)
            out.append((film, cnt, integ.counters(), integ.readbackViewSums(0), integ.readbackViewSums(1)))
    _same(out[0][1], out[1][1])
    _same(out[0][2], out[1][2])
    for i in (0, 3, 4):
        # float64 sums of a few float32 radiances per pixel in any order
        assert np.allclose(out[0][i], out[1][i], rtol=1e-14, atol=0) and out[0][i].any()


@pytest.mark.parametrize("width", [4, 8], ids=["bvh4", "bvh8"])
def test_timed_guided_render_records_the_same(width):
    desc = scenes.make_c3(width=96, height=64, spp=2, cell=0.5, n_props=8, prop_subdiv=1, hdri_w=256, hdri_h=128,
                          max_depth=6)
    out = []
    with Integrator.createIntegrator(IntegratorType.WavefrontPathTracing, 96, 64) as integ:
        integ.setBVHWidth(width)
        upload_scene(integ, desc)
        for timed in (True, False):
            integ.setTiming(timed)
            integ.guideReset(17)
            integ.setGuide(True, bsdf_fraction=0.5, train=1, record_paths=2 * 96 * 64, batch_size=32768, steps_per_batch=1)
            integ.resetIterationIndex()
            integ.render(2)
            cnt = integ.counters()
            V, E, smp = integ.guideRecords()
            out.append((cnt, integ.readbackSums(), V, E, smp, integ.guideStats()["last_count"]))
            integ.setGuide(False)
    a, b = out
    _same(a[0], b[0])
    assert np.allclose(a[1], b[1], rtol=1e-14, atol=0) and a[1].any()
    # few of the room's paths find the window: 2 samples a pixel give hundreds
    n = a[5]
    assert np.any(a[3]) and n == b[5] > 100
    for i, m in ((2, None), (3, None), (4, n)):
        assert np.array_equal(a[i][:m].view(np.uint32), b[i][:m].view(np.uint32)), i
