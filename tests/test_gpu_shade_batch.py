"""The shading batch that a launch chooses by the frame's samples, scene kind
and size changes when a wave shades, never what a pixel is: frames on both
sides of each edge of the rule and a batch, at the default and at fixed
shading batches, bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

# below and above two pixels per lane (524,288 on 256 CUs), 8 and 9 samples,
# 10 to 16 (longest tiles first)
FRAMES = [(300, 200, 8), (1030, 520, 1), (1030, 520, 8), (1030, 520, 9), (1030, 520, 15), (1030, 520, 16)]


def _render(rtx, s, lps, batched):
    out = []
    Ls = [rtx.Launcher(s, lp) for lp in lps]
    if batched:
        b = rtx.Batch(s, lps, use_graph=False)
        b.launch()
        b.free()
    else:
        for L in Ls:
            L.ignite()
    for L in Ls:
        out += [L.raw_rgb(), L.rays_per_pixel()]
        L.free()
    return out


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("batched", [False, True])
def test_frames_do_not_depend_on_the_shading_batch(rtx, two_level, batched):
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=6, half=4, level=2, two_level=two_level)
    s.load()
    h = s.build()
    try:
        def lps():
            r = []
            for w, hh, spp in FRAMES:
                lp = rtx.LpGeneral()
                lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, hh, spp, 10, h
                lp.camera = rtx.Camera().set((13, 2, 3), (0, 0, 0), (0, 1, 0), 20.0, w / hh, 0.1, 10.0).c
                r.append(lp)
            return r
        old = s.tuning()["shade_batch"]
        want = _render(rtx, s, lps(), batched)
        for sb in (1, 33, 64):
            say("shading batch %d, %s" % (sb, "two-level" if two_level else "flat"))
            s.tuning(shade_batch=sb)
            for a, b in zip(want, _render(rtx, s, lps(), batched)):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        s.tuning(shade_batch=old)
        for a, b in zip(want, _render(rtx, s, lps(), batched)):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        s.close()
