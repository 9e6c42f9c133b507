"""The first query of a context: what it allocates, and its answer.  A query
over a scene whose traversal fits the stack in LDS, and every pick, take no
device memory; deeper scenes get their overflow area and answer alike."""
from ctypes import byref

import numpy as np
import pytest
import torch

from test_gpu_parity import say
from test_gpu_small_trees import _build, _rays_at, _soup

pytestmark = pytest.mark.gpu


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("two_level", [False, True])
def test_first_query_of_a_shallow_scene_allocates_nothing(rtx, two_level):
    tris = _soup(300, 3)
    s = _build(rtx, tris, two_level)
    try:
        n = 5000
        rays = torch.from_numpy(_rays_at(tris, n, 4)).cuda()
        hits = torch.zeros((n, 8), dtype=torch.int32, device="cuda")
        before = _free()
        assert rtx.lib().rtx_trace(s.ctx, s.handle, rays.data_ptr(), n, hits.data_ptr(), None) == 0
        after = _free()
        say("%s, wide depth %d: %d bytes" % ("two-level" if two_level else "flat", s.stats()["wide_depth"], before - after))
        assert after == before
        assert torch.isfinite(hits.view(torch.float32)[:, 0]).float().mean() > 0.5
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("level", [1, 4])
def test_first_pick_allocates_nothing(rtx, level, two_level):
    """Picks as the first calls of a context, against closest hits of the
    same things seen through a pinhole."""
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=3, half=6, level=level, two_level=two_level)
    s.load()
    s.build()
    try:
        lp = rtx.LpGeneral()
        w, h = 160, 90
        lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, h, 1, 16, s.handle
        lp.camera = rtx.Camera().set((13, 2, 3), (0, 0, 0), (0, 1, 0), 20.0, w / h, 0.0, 10.0).c
        pick = torch.zeros(1, dtype=torch.int32, device="cuda")
        lp.picker, lp.pick_id = True, pick.data_ptr()
        got = []
        before = _free()
        for y in range(5, h, 12):
            for x in range(3, w, 13):
                lp.pick_x, lp.pick_y = x, y
                rtx._capi.call("rtx_launch", s.ctx, byref(lp), 1, None)
                got.append(int(pick.item()) & 0xFFFFFFFF)
        assert _free() == before
        say("level %d, %s: %d picks" % (level, "two-level" if two_level else "flat", len(got)))
        # an ordinary launch and a query allocate the overflow area; picks stay the same
        L = rtx.Launcher(s, lp)
        lp.picker = False
        L.ignite()
        lp.picker, lp.pick_id = True, pick.data_ptr()
        again = []
        for y in range(5, h, 12):
            for x in range(3, w, 13):
                lp.pick_x, lp.pick_y = x, y
                L.ignite(once=True)
                again.append(int(pick.item()) & 0xFFFFFFFF)
        L.free()
        assert got == again
        # the ids of the pixel centres' rays: equal but where the jitter crosses an outline
        c = lp.camera
        rays = np.zeros((len(got), 8), np.float32)
        k = 0
        for y in range(5, h, 12):
            for x in range(3, w, 13):
                u, v = 2 * (x + .5) / w - 1, 2 * (y + .5) / h - 1
                rays[k, 0:3] = tuple(c.eye)
                rays[k, 4:7] = u * np.array(tuple(c.wvec)) + v * np.array(tuple(c.hvec)) - np.array(tuple(c.dvec))
                k += 1
        rays[:, 3], rays[:, 7] = 1e-3, 1e16
        ids = s.trace(rays)["instance_id"]
        assert (ids == np.array(got, np.uint32)).mean() > 0.85
    finally:
        s.close()
