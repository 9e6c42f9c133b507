"""Scene builds share a device's workspace: its memory is used again by the
next build, which may be larger or smaller, and a build beside another one
takes memory of its own.  Levels are launched ahead of their counts, for the
most tasks that they can have.  So a scene's tree must not depend on what was
built before it or is built beside it: its statistics and hits are bit for bit
those of the same scene built first.
"""
import threading

import numpy as np
import pytest

from test_gpu_parity import say
from test_gpu_small_trees import _build, _rays_at, _soup

pytestmark = pytest.mark.gpu

# a leaf at the root, one split, the sizes of a thread's, a wave's and a
# block's task and one past them, a level spread over many blocks
SIZES = (1, 2, 9, 17, 65, 257, 4097, 70001)


def _mixed(rtx, parts):
    """A two-level scene of several trees (their results stay in the workspace)."""
    s = rtx.Scene()
    s.build_mode(rtx.Scene.TWO_LEVEL)
    for t in parts:
        v = t.reshape(-1, 3)
        m = s.add((v, np.arange(len(v), dtype=np.uint32).reshape(-1, 3)))
        for k in range(3):
            x = np.eye(3, 4, dtype=np.float32)
            x[0, 3] = 3.0 * k
            s.set(s.add(rtx.Thing.diffuse((.5, .5, .5)), m), x)
    s.build()
    return s


def _seen(s, rays):
    h = s.trace(rays)
    st = s.stats()
    return ([h[k].tobytes() for k in ("t", "prim", "instance_id")],
            [st[k] for k in ("num_nodes", "num_leaves", "max_depth", "max_leaf", "wide_nodes")])


def _scene(rtx, n, kind):
    if kind == "mixed":
        return _mixed(rtx, [_soup(k, 50 + k) for k in (1, n, 3)])
    return _build(rtx, _soup(n, 50 + n), kind == "two-level")


@pytest.mark.parametrize("kind", ["flat", "two-level", "mixed"])
def test_order_of_builds(rtx, kind):
    rays = {n: _rays_at(_soup(n, 50 + n), 3000, n) for n in SIZES}
    first = {}
    for n in SIZES:                       # every build is the largest so far
        say("%s build of %d triangles, growing" % (kind, n))
        s = _scene(rtx, n, kind)
        first[n] = _seen(s, rays[n])
        s.close()
    for n in SIZES[::-1] + SIZES[::2]:    # and after larger and smaller ones
        say("%s build of %d triangles, again" % (kind, n))
        s = _scene(rtx, n, kind)
        assert _seen(s, rays[n]) == first[n], n
        s.close()


def test_builds_beside_each_other(rtx):
    sizes = SIZES[2:]
    rays = {n: _rays_at(_soup(n, 50 + n), 3000, n) for n in sizes}
    want = {}
    for n in sizes:
        s = _scene(rtx, n, "flat")
        want[n] = _seen(s, rays[n])
        s.close()
    wrong = []

    def work(order):
        try:
            for n in order:
                s = _scene(rtx, n, "flat")
                if _seen(s, rays[n]) != want[n]:
                    wrong.append(n)
                s.close()
        except Exception as e:   # shown by the main thread
            wrong.append(e)

    say("builds in 3 threads")
    th = [threading.Thread(target=work, args=(o,)) for o in (sizes, sizes[::-1], sizes[::2])]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not wrong
