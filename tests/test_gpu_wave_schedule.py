"""The schedule that one wavefront makes of up to 64 experts (grouped_gemm.hip, wave_schedule): its records against the host
mirror's, and the tiles handed out, first ones and drawn ones, against the same call with a caller's workspace, whose records another
kernel writes.  Numbers of experts around the eight keys of a step and the 64 lanes, ties, empty experts, one kind only."""
import ctypes

import numpy as np
import pytest
import torch

from tests.test_gpu_one_launch import _mm, _read_stream_workspace

pytestmark = pytest.mark.gpu


def _rows(experts, kind):
    rng = np.random.default_rng(experts)
    if kind == "ties":
        return [(0, 70, 5, 70, 64, 65)[i % 6] for i in range(experts)]
    high = {"light": 65, "heavy": 400, "mixed": 130}[kind]
    return [int(v) for v in rng.integers(66 if kind == "heavy" else 0, high, size=experts)]


@pytest.mark.parametrize("kind", ["light", "heavy", "mixed", "ties"])
@pytest.mark.parametrize("experts", [1, 7, 8, 9, 16, 63, 64])
def test_records_and_tiles(esmoe, experts, kind):
    from expert_specialization_moe_amd import _native
    from expert_specialization_moe_amd import workloads as W

    lib, n, k = _native.lib, 640, 256
    rows = _rows(experts, kind)
    if not sum(rows):
        rows[0] = 3
    print(f"{kind} E={experts} rows={rows}", flush=True)
    mx = experts % 2 == 0
    prob = W.Problem("wave", n, k, rows, kind="mxfp8" if mx else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if mx else W.make_fp8_blockwise_operands)(prob, "cuda", seed=experts, weight_std=0.05)
    words = lib.esmoe_gemm_workspace_bytes(experts) // 4
    ws = torch.full((words,), -1, dtype=torch.int32, device="cuda").view(torch.uint8)
    name = "mx" if mx else "fp8"
    want = _mm(_native, ops, name, ws, torch.full_like(ops["output"], float("nan")))
    got = _mm(_native, ops, name, None, torch.full_like(ops["output"], float("nan")))
    assert not torch.isnan(got).any()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    host = np.zeros(words, dtype=np.int32)
    ps = np.array([[m, n, k] for m in rows], dtype=np.int32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    assert lib.esmoe_host_schedule(ptr(ps), experts, n, 0, int(mx), ptr(host)) == 0, _native.last_error()
    dev, first = _read_stream_workspace(_native, words), 64 + 32 * 8
    assert np.array_equal(dev[first:first + 4 * (experts + 1)], host[first:first + 4 * (experts + 1)])
    assert not dev[[16, 32] + [64 + 32 * x for x in range(8)]].any()   # every counter is back at zero
