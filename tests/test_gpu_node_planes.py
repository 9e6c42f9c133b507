"""Closest hits where the 4-wide nodes' 16-bit planes and the slab test's
margins matter: rays that run within the faces of boxes (parallel to an axis,
through the vertices and edges of a grid), scenes of very small and very large
extent, tiny triangles beside huge ones, and a two-level scene refitted far
beyond the extent it was built with."""
import numpy as np
import pytest

from test_gpu_parity import say
from test_gpu_small_trees import _build, _rays_at, _soup

pytestmark = pytest.mark.gpu


def _grid(n, axis, at):
    """n x n unit squares, two triangles each, in the plane axis = at, corner at the origin."""
    p = np.array([[[x, y], [x + 1, y], [x + 1, y + 1], [x, y], [x + 1, y + 1], [x, y + 1]]
                  for x in range(n) for y in range(n)], np.float32).reshape(-1, 2)
    v = np.full((len(p), 3), at, np.float32)
    v[:, (axis + 1) % 3] = p[:, 0]
    v[:, (axis + 2) % 3] = p[:, 1]
    return v.reshape(-1, 3, 3)


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("shift,at", [(0., 0.), (-5., 0.25), (96., 3.), (-1000., -512.)])
def test_rays_within_box_faces(rtx, axis, shift, at, two_level):
    """Every ray parallel to the grid's normal through an interior vertex, edge
    midpoint or face centre hits it, at the exact distance: 4 to the plane
    along unit directions, all coordinates exact in FP32."""
    n = 9
    tris = _grid(n, axis, at)
    tris[:, :, (axis + 1) % 3] += np.float32(shift)
    tris[:, :, (axis + 2) % 3] -= np.float32(shift)
    g = np.arange(2, 2 * n - 1) / 2.0           # 1 .. n - 1 by halves
    a, b = (x.ravel() for x in np.meshgrid(g, g))
    rays = np.zeros((2 * len(a), 8), np.float32)
    rays[:, (axis + 1) % 3] = np.concatenate([a, a]) + shift
    rays[:, (axis + 2) % 3] = np.concatenate([b, b]) - shift
    rays[:len(a), axis] = at + 4
    rays[len(a):, axis] = at - 4
    rays[:len(a), 4 + axis] = -1
    rays[len(a):, 4 + axis] = 1
    rays[:, 3] = 1e-3
    rays[:, 7] = 1e16
    say("grid in the plane of axis %d, shift %g, %s" % (axis, shift, "two-level" if two_level else "flat"))
    s = _build(rtx, tris, two_level)
    try:
        t = s.trace(rays)["t"]
        assert (t == np.float32(4)).all()
    finally:
        s.close()


@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("log2", [-30, -12, 12, 24])
def test_hits_do_not_depend_on_the_scale(rtx, log2, two_level):
    """A scene and its rays scaled by a power of two: the same hits, bit for
    bit (every FP32 operation of the intersection scales exactly)."""
    tris = _soup(60, 77)
    rays = _rays_at(tris, 6000, 78)
    got = []
    for k in (0, log2):
        f = np.float32(2.0 ** k)
        r = rays.copy()
        r[:, 0:3] *= f
        r[:, 4:7] *= f
        say("scale 2^%d, %s" % (k, "two-level" if two_level else "flat"))
        s = _build(rtx, tris * f, two_level)
        try:
            got.append(s.trace(r))
        finally:
            s.close()
    assert np.isfinite(got[0]["t"]).mean() > 0.5
    for key in ("t", "u", "v", "prim", "instance_id", "primitive_index"):
        assert np.array_equal(got[0][key], got[1][key]), key


@pytest.mark.parametrize("two_level", [False, True])
def test_tiny_triangles_beside_huge_ones(rtx, orc, two_level):
    """A cloud of triangles of size 0.01 ten units off the origin, between
    triangles of size 10^5: ids against the FP64 brute force where decidable."""
    tiny = _soup(400, 5) * np.float32(0.05) + np.float32(10)
    huge = _soup(6, 6) * np.float32(1e5) - np.float32(3e5)
    tris = np.concatenate([tiny, huge]).astype(np.float32)
    g = np.random.default_rng(9)
    n = 6000
    rays = _rays_at(tiny, n, 10)
    o = g.normal(size=(n, 3))
    o = 10 + 1.0 * o / np.linalg.norm(o, axis=1)[:, None]
    k = g.integers(0, len(tiny), n)
    rays[:, 0:3] = o
    rays[:, 4:7] = tiny[k].astype(np.float64).mean(axis=1) - o
    rays[:, 3] = 1e-3
    say("tiny beside huge, %s" % ("two-level" if two_level else "flat"))
    s = _build(rtx, tris, two_level)
    try:
        world, _ = s.triangles()
        hits = s.trace(rays)
        gp = np.where(hits["instance_id"] == 0xFFFFFFFF, 0xFFFFFFFF, hits["prim"]).astype(np.uint32)
        ref = orc.closest_f64_brute(world, rays)
        ok = orc.decidable(ref, rays, world)
        say("decidable fraction %.4f" % ok.mean())
        assert ok.mean() > 0.5
        assert not (ok & (gp != ref["prim"])).any()
    finally:
        s.close()


def test_refit_beyond_the_built_extent(rtx):
    """Things moved 30 and 3000 extents apart by a refit hit like a fresh build."""
    mesh = (np.asarray(_soup(30, 21)).reshape(-1, 3), np.arange(90, dtype=np.uint32).reshape(-1, 3))
    g = np.random.default_rng(22)
    at = g.uniform(-2, 2, (12, 3)).astype(np.float32)

    def scene(f):
        s = rtx.Scene()
        s.build_mode(rtx.Scene.TWO_LEVEL)
        m = s.add(mesh)
        for k in range(len(at)):
            s.add(rtx.Thing.diffuse((.5, .5, .5)), m)
            place(s, k, f)
        s.build()
        return s

    def place(s, k, f):
        x = np.zeros((3, 4), np.float32)
        x[:, :3] = np.eye(3)
        x[:, 3] = at[k] * np.float32(f)
        s.set(k, x)

    s = scene(1)
    try:
        for f in (30, 3000):
            for k in range(len(at)):
                place(s, k, f)
            s.update(s.handle)
            rays = np.zeros((4000, 8), np.float32)
            o = g.normal(size=(len(rays), 3)) * f
            k = g.integers(0, len(at), len(rays))
            rays[:, 0:3] = o
            rays[:, 4:7] = at[k] * f + g.uniform(-1, 1, (len(rays), 3)) - o
            rays[:, 3] = 1e-3
            rays[:, 7] = 1e16
            say("refit to %d times the extent" % f)
            a = s.trace(rays)
            fresh = scene(f)
            try:
                b = fresh.trace(rays)
            finally:
                fresh.close()
            assert np.isfinite(a["t"]).mean() > 0.1
            for key in ("t", "u", "v", "prim", "instance_id"):
                assert np.array_equal(a[key], b[key]), key
    finally:
        s.close()
