"""The device memory that builds keep for the next one: given back on request
and with the last context, shrunk when builds have long been small; builds
and hits do not depend on it."""
import numpy as np
import pytest
import torch

from test_gpu_parity import say
from test_gpu_small_trees import _build, _rays_at, _soup

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.fixture(autouse=True, scope="module")
def _first_kernels(rtx):
    """The process's first kernels load code and take scratch memory for good."""
    for n in (64, 1 << 19):
        _build_and_close(rtx, _soup(n, 1), _rays_at(_soup(64, 1), 4000, 2))


def _build_and_close(rtx, tris, rays=None):
    s = _build(rtx, tris, False)
    try:
        return s.trace(rays)["t"] if rays is not None else None
    finally:
        s.close()


def test_kept_memory_is_given_back(rtx):
    tris = _soup(1 << 19, 11)
    rays = _rays_at(tris, 4000, 12)
    holder = rtx.Scene()                      # a context that outlives the builds
    try:
        holder.trim()
        start = _free()
        first = _build_and_close(rtx, tris, rays)
        kept = start - _free()
        say("kept after a build of %d triangles: %d MiB" % (len(tris), kept // MIB))
        assert kept > 64 * MIB
        holder.trim()
        assert start - _free() < 4 * MIB
        holder.trim()                         # nothing left to give back
        # a build after it takes and keeps the same again, with the same hits
        assert np.array_equal(_build_and_close(rtx, tris, rays), first)
        assert abs(start - _free() - kept) < 4 * MIB
    finally:
        holder.close()


def test_kept_memory_shrinks_after_small_builds(rtx):
    big, small = _soup(1 << 19, 11), _soup(64, 13)
    rays = _rays_at(small, 2000, 14)
    holder = rtx.Scene()
    try:
        holder.trim()
        start = _free()
        want = _build_and_close(rtx, small, rays)
        _build_and_close(rtx, big)
        kept = start - _free()
        for k in range(7):
            assert np.array_equal(_build_and_close(rtx, small, rays), want)
        assert start - _free() > kept // 2    # a few small builds keep the block
        _build_and_close(rtx, big)
        for k in range(8):
            assert np.array_equal(_build_and_close(rtx, small, rays), want)
        left = start - _free()
        say("kept %d MiB, after eight small builds %d MiB" % (kept // MIB, left // MIB))
        assert left < 8 * MIB
    finally:
        holder.close()
