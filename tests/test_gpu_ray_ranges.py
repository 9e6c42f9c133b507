"""Closest hits over the whole range of what a ray may hold: negative tmin
(lines and segments that begin behind the origin), tmin just below the hit
(stepping through hits), unbounded tmax over tiny scenes, and direction
components that are subnormal, zero of either sign or far below the others.
Flat and two-level layouts."""
import numpy as np
import pytest

from test_gpu_node_planes import _grid
from test_gpu_parity import say
from test_gpu_small_trees import _build, _rays_at, _soup

pytestmark = pytest.mark.gpu

INF = np.float32(np.inf)


def _layers(n, axis, at):
    return np.concatenate([_grid(n, axis, z) for z in at])


def _axis_rays(n, axis, sign=1):
    """Rays along the axis from its plane 0, through interior vertices, edge
    midpoints and face centres of an n x n grid."""
    g = np.arange(2, 2 * n - 1) / 2.0
    a, b = (x.ravel() for x in np.meshgrid(g, g))
    rays = np.zeros((len(a), 8), np.float32)
    rays[:, (axis + 1) % 3] = a
    rays[:, (axis + 2) % 3] = b
    rays[:, 4 + axis] = sign
    rays[:, 3] = 1e-3
    rays[:, 7] = 1e16
    return rays


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_lines_through_layers(rtx, axis, two_level):
    """The first layer above tmin is hit, at its exact distance, whichever
    side of the origin it is on; a segment that ends before it hits nothing."""
    at = np.array([-9., -6.5, -4., -1.5, 2., 4.5, 5., 8.])
    s = _build(rtx, _layers(6, axis, at), two_level)
    try:
        for sign in (1, -1):
            rays = _axis_rays(6, axis, sign)
            t = np.sort(at * sign)
            for tmin in (-INF, -1e16, -1000., -10., -7., -5., -4., -1., -1e-3, 0., 3.):
                for tmax in (-6., -1.25, 3., 4.75, 10., 1e16, INF):
                    rays[:, 3], rays[:, 7] = tmin, tmax
                    want = t[(t > np.float32(tmin)) & (t <= np.float32(tmax))]
                    want = np.float32(want[0]) if len(want) else INF
                    got = s.trace(rays)["t"]
                    say("axis %d, direction %d, tmin %g, tmax %g: %g" % (axis, sign, tmin, tmax, want))
                    assert (got == want).all()
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("n", [3, 40, 600])
def test_lines_through_a_soup(rtx, orc, n, two_level):
    """Lines with negative tmin against the FP64 brute force, which tests every triangle."""
    tris = _soup(n, 300 + n)
    s = _build(rtx, tris, two_level)
    try:
        for k, tmin in enumerate((-0.25, -1., -3., -1e16)):
            rays = _rays_at(tris, 6000, 40 + k)
            # from inside and beside the soup; the hit may be at a negative distance
            rays[:, 0:3] += (rays[:, 4:7] * np.random.default_rng(k).uniform(0, 2, (len(rays), 1))).astype(np.float32)
            rays[:, 3] = tmin
            ref = orc.closest_f64_brute(tris, rays)
            ok = orc.decidable(ref, rays, tris)
            hits = s.trace(rays)
            gp = np.where(hits["instance_id"] == 0xFFFFFFFF, 0xFFFFFFFF, hits["prim"]).astype(np.uint32)
            neg = (hits["t"] < 0).mean()
            say("%d triangles, tmin %g: %.2f of the hits behind the origin, %.3f decidable" % (n, tmin, neg, ok.mean()))
            assert neg > 0.02 and ok.mean() > 0.5
            assert not (ok & (gp != ref["prim"])).any()
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
def test_tmin_just_below_the_hit(rtx, two_level):
    """A ray whose tmin lies between nothing and its hit finds the hit again,
    also through the edges and vertices that several boxes share."""
    g = np.random.default_rng(5)
    n = 24
    tris = _grid(n, 2, 0.)
    tris[:, :, 2] = np.float32(0.4) * np.sin(3 * tris[:, :, 0]) * np.cos(2 * tris[:, :, 1])
    s = _build(rtx, tris, two_level)
    try:
        m = 40000
        tri = tris[g.integers(0, len(tris), m)].astype(np.float64)
        w = g.integers(0, 3, (m, 3)).astype(np.float64)       # vertices, edge and inner points
        w[w.sum(1) == 0] = 1.
        p = (w[:, :, None] * tri).sum(1) / w.sum(1)[:, None]
        rays = np.zeros((m, 8), np.float32)
        rays[:, 0:3] = p + g.normal(size=(m, 3)) * [8, 8, 3] + [0, 0, 9]
        rays[:, 4:7] = (p - rays[:, 0:3]) * g.uniform(0.1, 3, (m, 1))
        rays[:, 7] = 1e16
        first = s.trace(rays)
        t = first["t"]
        assert np.isfinite(t).mean() > 0.9
        for f in (0.5, 0.9, 0.99, 0.999, 0.9999, 0.99999, 1.):
            rays[:, 3] = np.nextafter(t, np.float32(0)) if f == 1. else t * np.float32(f)
            rays[~np.isfinite(t), 3] = 0.
            again = s.trace(rays)
            say("tmin at %g of the hit" % f)
            for key in ("t", "prim"):
                assert np.array_equal(again[key], first[key]), key
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("tiny", [-0., 1e-44, -1e-41, 1e-39, -3e-39, 1e-36, -1e-30, 1e-26, 1e-20])
def test_tiny_direction_components(rtx, axis, tiny, two_level):
    """Components whose reciprocal is infinite or huge: the ray is parallel to the axis."""
    s = _build(rtx, _layers(6, axis, (-4., 4., 4.5)), two_level)
    try:
        rays = np.concatenate([_axis_rays(6, axis, 1), _axis_rays(6, axis, -1)])
        for k in ((1,), (2,), (1, 2)):
            for j in k:
                rays[:, 4 + (axis + j) % 3] = tiny
            say("axis %d, component %g" % (axis, tiny))
            assert (s.trace(rays)["t"] == np.float32(4)).all()
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("log2", [-90, -70, -50, 40])
def test_short_and_long_directions(rtx, log2, two_level):
    """A direction of length 2^k along an axis: the distance is 4 / 2^k."""
    for axis in (0, 1, 2):
        s = _build(rtx, _layers(6, axis, (-4., 4., 4.5)), two_level)
        try:
            rays = np.concatenate([_axis_rays(6, axis, 1), _axis_rays(6, axis, -1)])
            rays[:, 4:7] *= np.float32(2.0 ** log2)
            rays[:, 3], rays[:, 7] = 0., INF
            say("axis %d, direction 2^%d" % (axis, log2))
            assert (s.trace(rays)["t"] == np.float32(4 * 2.0 ** -log2)).all()
        finally:
            s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("log2", [-36, -30, 0, 20])
def test_unbounded_rays_of_unit_direction(rtx, log2, two_level):
    """tmax unbounded and the direction of length one, whatever the extent of
    the scene: the hits of the same rays with a tmax of its size."""
    f = np.float32(2.0 ** log2)
    tris = _soup(200, 7) * f
    s = _build(rtx, tris, two_level)
    try:
        rays = _rays_at(tris / f, 20000, 8)
        rays[:, 0:3] *= f
        rays[:, 4:7] /= np.linalg.norm(rays[:, 4:7], axis=1)[:, None]
        rays[:, 3], rays[:, 7] = 0., 8 * f
        want = s.trace(rays)
        assert np.isfinite(want["t"]).mean() > 0.5
        for tmax in (1e16, 1e30, np.finfo(np.float32).max, INF):
            rays[:, 7] = tmax
            say("scale 2^%d, tmax %g" % (log2, tmax))
            got = s.trace(rays)
            for key in ("t", "prim"):
                assert np.array_equal(got[key], want[key]), key
    finally:
        s.close()
