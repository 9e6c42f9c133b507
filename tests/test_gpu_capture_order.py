"""Frames and gradient launches that are rendered in probe order, captured
into a HIP graph in a context that has not allocated the order's arrays: the
capture takes them, in slot order, and every replay gives the eager pixels."""
import ctypes

import numpy as np
import pytest
import torch

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _scene(rtx):
    from rtxplay_amd.scene import RTOWScene
    s = RTOWScene(seed=5, half=5, level=2)
    s.load()
    s.build()
    return s


def _lp(rtx, s, w, h, spp):
    lp = rtx.LpGeneral()
    lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, h, spp, 6, s.handle
    lp.camera = rtx.Camera().set((13, 2, 3), (0, 0, 0), (0, 1, 0), 20.0, w / h, 0.1, 10.0).c
    out = torch.zeros((h, w, 3), device="cuda"), torch.zeros((h, w), dtype=torch.int32, device="cuda")
    lp.rawRGB, lp.rpp = out[0].data_ptr(), out[1].data_ptr()
    return lp, out


@pytest.mark.parametrize("spp", [10, 16])
def test_ordered_frame_captured_first(rtx, spp):
    from rtxplay_amd._capi import byref, call
    s = _scene(rtx)
    try:
        small, _ = _lp(rtx, s, 64, 40, 1)
        call("rtx_launch", s.ctx, byref(small), 0, _stream())
        lp, (img, rpp) = _lp(rtx, s, 1100, 600, spp)      # two pixels per lane and more
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call("rtx_launch", s.ctx, byref(lp), 0, _stream())
        got = []
        for k in range(3):
            img.fill_(-1)
            rpp.fill_(-1)
            g.replay()
            torch.cuda.synchronize()
            got.append((img.clone(), rpp.clone()))
        img.fill_(-1)
        call("rtx_launch", s.ctx, byref(lp), 0, _stream())     # ordered now
        torch.cuda.synchronize()
        say("%d samples: %d rays" % (spp, int(rpp.sum())))
        for a, b in got:
            assert torch.equal(a, img) and torch.equal(b, rpp)
        del g
    finally:
        s.close()


def test_ordered_adjoint_captured_first(rtx):
    from rtxplay_amd._capi import byref, call
    s = _scene(rtx)
    try:
        n = len(s)
        d = torch.zeros((n, 4), device="cuda")
        small, (si, _) = _lp(rtx, s, 64, 40, 2)
        g0 = torch.ones_like(si)
        call("rtx_launch", s.ctx, byref(small), 0, _stream())
        call("rtx_launch_adjoint", s.ctx, byref(small), g0.data_ptr(), d.data_ptr(), _stream())
        lp, (img, _) = _lp(rtx, s, 480, 270, 16)          # more than two pixels per five lanes
        call("rtx_launch", s.ctx, byref(lp), 0, _stream())
        dl = torch.rand(img.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) + 0.5
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call("rtx_launch_adjoint", s.ctx, byref(lp), dl.data_ptr(), d.data_ptr(), _stream())
        got = []
        for k in range(3):
            d.fill_(7)
            g.replay()
            torch.cuda.synchronize()
            got.append(d.cpu().numpy().astype(np.float64))
        call("rtx_launch_adjoint", s.ctx, byref(lp), dl.data_ptr(), d.data_ptr(), _stream())
        torch.cuda.synchronize()
        want = d.cpu().numpy().astype(np.float64)
        say("gradient of %d things, largest %g" % (n, np.abs(want).max()))
        # the same terms summed by float atomics in another order: 16 x 129600
        # x 6 = 1.2e7 of one entry at most, roundings of 2^-24 of the partial
        # sum each, sqrt(1.2e7) * 2^-24 = 2e-4 of it; ten times that, and for
        # fuzz, whose terms cancel, as much of a tenth of the largest entry
        for a in got:
            assert np.allclose(a, want, rtol=2e-3, atol=2e-3 * np.abs(want).max() / 10)
        del g
    finally:
        s.close()
