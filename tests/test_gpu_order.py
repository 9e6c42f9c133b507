"""Ordered frames (10 samples and more, two pixels per lane of the persistent
grid and more): a probe orders the tiles by the cost of their neighbourhoods
and gives the most expensive pixels to waves of 8, 16 or 32 lanes.  No pixel
may be left out, taken twice or changed: frames with ragged edges and every
shape of tile against the batch launch, which takes tiles in order, bit for
bit; the adjoint's sums for tiles of other shapes, which are replayed in
another order, against each other.
"""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def _lp(rtx, h, w, hh, spp, depth, cam):
    lp = rtx.LpGeneral()
    lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, hh, spp, depth, h
    lp.camera = rtx.Camera().set(cam, (0, 0, 0), (0, 1, 0), 20.0, w / hh, 0.1, 10.0).c
    return lp


# (w, h, tile width, blocks per CU): 524,288 pixels are two per lane
FRAMES = [(1024, 512, 8, 4), (1023, 515, 8, 4), (1301, 409, 1, 4), (411, 1283, 64, 4), (2049, 257, 16, 2),
          (737, 731, 2, 1), (1031, 1021, 8, 3)]


@pytest.mark.parametrize("two_level", [False, True])
def test_ordered_frames_equal_batch_frames(rtx, two_level):
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=9, half=4, level=2, two_level=two_level)
    s.load()
    h = s.build()
    old = s.tuning()
    try:
        # from afar most of the frame is sky (few expensive pixels, many narrow waves); from near none is
        for cam in ((13, 2, 3), (40, 6, 9), (2.5, .6, 1.)):
            for w, hh, tw, bpc in FRAMES:
                say("%dx%d, tiles of width %d, %d blocks per CU, %s" % (w, hh, tw, bpc,
                                                                       "two-level" if two_level else "flat"))
                s.tuning(tile_w=tw, blocks_per_cu=bpc)
                got = []
                for batched in (False, True):
                    lp = _lp(rtx, h, w, hh, 10, 12, cam)
                    L = rtx.Launcher(s, lp)
                    if batched:
                        b = rtx.Batch(s, [lp], use_graph=False)
                        b.launch()
                        b.free()
                    else:
                        L.ignite()
                    got.append((L.raw_rgb(), L.rays_per_pixel(), L.normals(), L.albedos()))
                    L.free()
                assert (got[0][1] >= 10).all()
                for a, b in zip(*got):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    finally:
        s.tuning(tile_w=old["tile_w"], blocks_per_cu=old["blocks_per_cu"])
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
def test_ordered_adjoint_does_not_depend_on_the_tiles(rtx, two_level):
    import torch
    from rtxplay_amd.diff import DiffRender, material_params
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=9, half=4, level=2, two_level=two_level)
    s.load()
    h = s.build()
    old = s.tuning()
    try:
        for w, hh in ((431, 245), (977, 539)):
            grads = []
            for tw in (8, 1, 64):
                say("%dx%d, tiles of width %d, %s" % (w, hh, tw, "two-level" if two_level else "flat"))
                s.tuning(tile_w=tw)
                p = material_params(s.things_spec).to("cuda").requires_grad_(True)
                img = DiffRender(s, _lp(rtx, h, w, hh, 16, 8, (13, 2, 3)))(p)
                g = torch.linspace(.5, 1.5, img.numel(), device="cuda").reshape(img.shape)
                (img * g).sum().backward()
                grads.append(p.grad.double().cpu().numpy())
            # float sums of up to 1e7 terms of mostly one sign in different orders: 2^-24 * sqrt(1e7)
            # = 2e-4 of the sum
            for k in grads[1:]:
                assert np.abs(k - grads[0]).max() < 2e-4 * np.abs(grads[0]).max()
    finally:
        s.tuning(tile_w=old["tile_w"])
        s.close()


def test_noalloc_frame_beyond_the_static_tiles_renders_in_slot_order(rtx):
    """270,000 tiles of 64x1 with 2 pixels each, 10 samples: more than the static
    scratch orders, and fewer samples than are refused."""
    import ctypes
    import torch
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=9, half=4, level=2)
    s.load()
    h = s.build()
    old = s.tuning()
    try:
        s.tuning(tile_w=64)
        got = []
        for entry in ("rtx_launch", "rtx_launch_noalloc"):
            say(entry)
            lp = _lp(rtx, h, 2, 270000, 10, 6, (13, 2, 3))
            img = torch.zeros((270000, 2, 3), device="cuda")
            c = lp if isinstance(lp, ctypes.Structure) else lp.c
            c.rawRGB = img.data_ptr()
            st = getattr(rtx.lib(), entry)(s.ctx, ctypes.byref(c), 0, None)
            assert st == 0, rtx.lib().rtx_last_error()
            torch.cuda.synchronize()
            got.append(img.cpu().numpy())
        assert got[0].max() > 0
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    finally:
        s.tuning(tile_w=old["tile_w"])
        s.close()
