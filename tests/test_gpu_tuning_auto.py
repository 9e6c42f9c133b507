"""Launch tuning: every shading batch from 1 to 64 can be chosen, 40 (the
default) among them, and the library's own choice can be had back."""
from ctypes import byref

import pytest

pytestmark = pytest.mark.gpu


def test_shading_batch_chosen_and_given_back(rtx):
    s = rtx.Scene()
    try:
        t = s.tuning()
        assert (t["shade_batch"], t["shade_auto"]) == (40, 1)
        # other fields leave the choice where it is
        t = s.tuning(tile_w=16)
        assert (t["shade_batch"], t["shade_auto"], t["tile_w"]) == (40, 1, 16)
        for sb in (40, 1, 64, 40):
            t = s.tuning(shade_batch=sb)
            assert (t["shade_batch"], t["shade_auto"]) == (sb, 0)
            assert s.tuning(tile_w=8)["shade_auto"] == 0
        old = s.tuning()
        t = s.tuning(shade_batch=40, shade_auto=1)
        assert (t["shade_batch"], t["shade_auto"]) == (40, 1)
        s.tuning(**{k: old[k] for k in ("shade_batch", "shade_auto")})
        assert s.tuning()["shade_auto"] == 0
    finally:
        s.close()


def test_structure_read_and_written_back(rtx):
    s = rtx.Scene()
    try:
        L, t = rtx.lib(), rtx._capi.TuningC()
        assert L.rtx_tuning_get(s.ctx, byref(t)) == 0
        assert L.rtx_tuning_set(s.ctx, byref(t)) == 0            # unchanged: still the library's choice
        assert s.tuning()["shade_auto"] == 1
        t.shade_batch = 24                                       # another value written into it is fixed
        assert L.rtx_tuning_set(s.ctx, byref(t)) == 0
        assert (s.tuning()["shade_batch"], s.tuning()["shade_auto"]) == (24, 0)
        t = rtx._capi.TuningC(shade_batch=40)                    # and so is 40 in a structure of its own
        assert L.rtx_tuning_set(s.ctx, byref(t)) == 0
        assert (s.tuning()["shade_batch"], s.tuning()["shade_auto"]) == (40, 0)
        t = rtx._capi.TuningC(shade_auto=1)
        assert L.rtx_tuning_set(s.ctx, byref(t)) == 0
        assert (s.tuning()["shade_batch"], s.tuning()["shade_auto"]) == (40, 1)
    finally:
        s.close()
