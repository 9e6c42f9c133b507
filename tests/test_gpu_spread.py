"""Frames whose pixels are spread over the waves (fewer than two per lane of
the persistent grid) against the batch launch, which takes tiles in order: the
same pixels, bit for bit, from one pixel to both sides of the rule's edges
(262,144 lanes on 256 CUs)."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 9), (7, 1, 5), (1, 65, 5), (63, 33, 4), (257, 129, 3), (512, 512, 1), (513, 511, 1), (1023, 511, 1),
         (1024, 512, 1), (1025, 515, 1)]


@pytest.mark.parametrize("two_level", [False, True])
def test_spread_frames_equal_batch_frames(rtx, two_level):
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=5, half=4, level=2, two_level=two_level)
    s.load()
    h = s.build()
    try:
        for w, hh, spp in SIZES:
            say("%dx%d, %d spp, %s" % (w, hh, spp, "two-level" if two_level else "flat"))
            got = []
            for batched in (False, True):
                lp = rtx.LpGeneral()
                lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, hh, spp, 12, h
                lp.camera = rtx.Camera().set((13, 2, 3), (0, 0, 0), (0, 1, 0), 20.0, w / hh, 0.1, 10.0).c
                L = rtx.Launcher(s, lp)
                if batched:
                    b = rtx.Batch(s, [lp], use_graph=False)
                    b.launch()
                    b.free()
                else:
                    L.ignite()
                got.append((L.raw_rgb(), L.rays_per_pixel(), L.normals(), L.albedos()))
                L.free()
            assert (got[0][1] >= spp).all()
            for a, b in zip(*got):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        s.close()
