"""Which light items of a fused MXFP8 launch go out as halves of 64 h columns, through the host mirror.  Halves last almost as long as whole
items, so they may only fill workgroups that would have nothing to do: where they make a second round of a launch that has one it
takes half as long again.  No GPU."""
import ctypes

import numpy as np
import pytest


def _tickets(rows, n, k, kind):
    """(light items, light tickets, heavy tiles or blocks)"""
    from expert_specialization_moe_amd import _native

    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    e = len(rows)
    ps = np.array([[m, n, k] for m in rows], dtype=np.int32)
    ws = np.zeros(_native.lib.esmoe_gemm_workspace_bytes(e) // 4, dtype=np.int32)
    assert _native.lib.esmoe_host_schedule(ptr(ps), e, n, 0, kind, ptr(ws)) == 0, _native.last_error()
    last = ws[64 + 32 * 8 + 4 * e:]
    return int(last[1]), int(ws[1]), int(last[0])


@pytest.mark.parametrize("k", [256, 640, 4096])
@pytest.mark.parametrize("items", [1, 2, 127, 128, 129, 133, 255, 256])
def test_a_launch_of_one_round_stays_one(esmoe, items, k):
    """256 workgroups: halves where all of them are first tickets, otherwise whole items."""
    assert _tickets([5] * items, 256, k, 3) == (items, 2 * items if items <= 128 else items, 0)


@pytest.mark.parametrize("heavy,light", [(1, 1), (18, 126), (66, 72), (100, 156)])
def test_beside_tall_tiles_of_the_same_round_items_stay_whole(esmoe, heavy, light):
    assert _tickets([100] * heavy + [9] * light, 256, 1280, 3) == (light, light, heavy)


@pytest.mark.parametrize("heavy,light,halves", [(0, 257, True), (0, 384, True), (0, 385, False), (0, 512, False), (48, 222, True), (60, 370, False),
                                                (256, 100, True), (256, 200, True), (700, 10, True)])
def test_the_end_of_a_longer_launch(esmoe, heavy, light, halves):
    """Halves, the last 128 items, where up to half a round is left or a round of tall tiles runs first; from K = 1024 on."""
    narrow = min(light, 128) if halves else 0
    assert _tickets([100] * heavy + [9] * light, 256, 1024, 3) == (light, light + narrow, heavy)
    assert _tickets([100] * heavy + [9] * light, 256, 896, 3) == (light, light, heavy)


def test_other_launches_are_as_they_were(esmoe):
    for items in (5, 200, 300):
        assert _tickets([5] * items, 256, 640, 2)[1] == items                          # FP8, fused: whole items
        assert _tickets([5] * items, 256, 128, 3)[1] == items                          # one K block
        assert _tickets([5] * items, 256, 640, 1)[1] == items + min(items, 128)        # plain: the last 128
