"""The 4-wide nodes' planes stay tight where things move far apart in a refit
and where a scene holds geometry that is minute beside its extent: node visits
per ray, counted, and the hits."""
import numpy as np
import pytest

from test_gpu_parity import say
from test_gpu_small_trees import _soup

pytestmark = pytest.mark.gpu


def _visits(rtx, s, eye, at, focus):
    """Node visits per ray of a small frame from eye towards at (no lens)."""
    lp = rtx.LpGeneral()
    lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = 96, 64, 2, 2, s.handle
    lp.camera = rtx.Camera().set(eye, at, (0, 1, 0), 30.0, 1.5, 0.0, focus).c
    L = rtx.Launcher(s, lp)
    try:
        nodes, _ = L.ignite_counted()
        return nodes.sum() / L.rays_per_pixel().sum()
    finally:
        L.free()


def _row(rtx, f, n=64):
    s = rtx.Scene()
    s.build_mode(rtx.Scene.TWO_LEVEL)
    m = s.add((np.asarray(_soup(200, 31)).reshape(-1, 3), np.arange(600, dtype=np.uint32).reshape(-1, 3)))
    for k in range(n):
        s.add(rtx.Thing.diffuse((.5, .5, .5)), m)
    _place(s, f, n)
    s.build()
    return s


def _place(s, f, n=64):
    for k in range(n):
        x = np.zeros((3, 4), np.float32)
        x[:, :3] = np.eye(3)
        x[:, 3] = np.array([k % 8 - 3.5, 0, k // 8 - 3.5]) * np.float32(3 * f)
        s.set(k, x)


def test_refit_far_apart_visits_as_few_nodes_as_a_build(rtx):
    """A grid of 64 things spread 40 and 4000 times as wide by a refit: the
    same arrangement as a fresh build, so about its node visits."""
    s = _row(rtx, 1)
    try:
        for f in (1, 40, 4000):
            _place(s, f)
            s.update(s.handle)
            fresh = _row(rtx, f)
            try:
                eye, at = (30. * f, 12. * f, 5. * f), (0., 0., 0.)
                a, b = _visits(rtx, s, eye, at, 30. * f), _visits(rtx, fresh, eye, at, 30. * f)
            finally:
                fresh.close()
            say("refit to %d times the spacing: %.2f visits per ray, fresh build %.2f" % (f, a, b))
            assert a <= 1.1 * b + 1.0
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
def test_minute_geometry_in_a_wide_scene(rtx, two_level):
    """4000 triangles within 2e-6 of the origin between triangles 1e6 away:
    rays at the cluster visit a few of its nodes, as in a scene of its own."""
    tiny = _soup(4000, 41) * np.array([1.5, 1.5, 1.5], np.float32)
    tiny = (tiny.mean(axis=1, keepdims=True) + (tiny - tiny.mean(axis=1, keepdims=True)) * np.float32(.1)) * np.float32(1e-6)
    far = _soup(8, 42) * np.float32(1e4) + np.float32(1e6)
    got = []
    for parts in ((tiny,), (tiny, far, -far)):
        s = rtx.Scene()
        if two_level:
            s.build_mode(rtx.Scene.TWO_LEVEL)
        for p in parts:
            m = s.add((p.reshape(-1, 3).astype(np.float32), np.arange(3 * len(p), dtype=np.uint32).reshape(-1, 3)))
            s.add(rtx.Thing.diffuse((.5, .5, .5)), m)
        s.build()
        try:
            got.append(_visits(rtx, s, (6e-6, 1e-6, 2e-6), (0., 0., 0.), 6e-6))
        finally:
            s.close()
    say("%s: %.1f visits per ray, alone %.1f" % ("two-level" if two_level else "flat", got[1], got[0]))
    assert got[1] <= 1.5 * got[0] + 10
