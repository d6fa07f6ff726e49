"""Records that the GEMM kernel's own schedule (self_schedule) and the schedule kernel write, against the host mirror's.

Light experts are placed by a count per row number, heavy ones by comparisons among themselves: the lists have ties, every row
number around the border of the two kinds, empty experts, one kind only, full wavefronts of experts and one expert more, and heavy lists
whose length is no multiple of four; order 2 ranks heavy experts the other way round and is set by a process-wide knob, so
it is left to the schedule kernel's own test of the host mirror.
"""
import ctypes

import numpy as np
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm, _read_stream_workspace

pytestmark = pytest.mark.gpu

LISTS = {
    "one_light": [1], "one_heavy": [65], "one_empty": [0, 1], "ties": [5, 5, 5, 0, 0, 5, 64, 64, 1],
    "border": [63, 64, 65, 66, 64, 65, 1, 0, 128, 65], "all_light": [(i * 7) % 65 for i in range(64)], "one_more": [(i * 11) % 65 for i in range(65)],
    "all_heavy": [65 + (i * 13) % 40 for i in range(67)], "every_third_heavy": [70 + i % 5 if i % 3 == 0 else i % 65 for i in range(200)],
    "two_heavy_of_512": [300 if i in (77, 401) else i % 4 for i in range(512)], "511": [(i * i) % 90 for i in range(511)],
}


@pytest.mark.parametrize("force_bm", [0, 64])
@pytest.mark.parametrize("name", list(LISTS))
def test_records_equal_the_host_mirror(esmoe, name, force_bm):
    from expert_specialization_moe_amd import _native, workloads as W

    rows, n, k = LISTS[name], 384, 128
    experts, total = len(rows), sum(rows)
    a = torch.zeros((total, k), device="cuda").to(torch.float8_e4m3fn)
    ops = dict(a=a, b_phys=torch.zeros((experts, n, k), device="cuda").to(torch.float8_e4m3fn),
               scales_a=torch.ones((total, 1), device="cuda"), scales_b_phys=torch.ones((experts, n // 128, 1), device="cuda"),
               problem_sizes=torch.tensor([[m, n, k] for m in rows], dtype=torch.int32, device="cuda"),
               expert_offsets=torch.tensor(W.offsets_of(rows), dtype=torch.int32, device="cuda"))
    out = torch.full((total, n), 3.0, dtype=torch.bfloat16, device="cuda")
    _mm(_native, ops, "fp8", None, out, force_bm)
    assert not out.any()   # every tile was handed out
    words = _native.lib.esmoe_gemm_workspace_bytes(experts) // 4
    dev = _read_stream_workspace(_native, words)
    host = np.zeros(words, dtype=np.int32)
    ps = np.array([[m, n, k] for m in rows], dtype=np.int32)
    rc = _native.lib.esmoe_host_schedule(ps.ctypes.data_as(ctypes.c_void_p), experts, n, force_bm, 0, host.ctypes.data_as(ctypes.c_void_p))
    assert rc == 0, _native.last_error()
    first = 64 + 32 * 8
    got, want = (v[first:first + 4 * (experts + 1)].reshape(-1, 4) for v in (dev, host))
    assert np.array_equal(got, want), np.flatnonzero((got != want).any(axis=1))


@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_both_schedules_note_where_an_experts_k_order_starts(esmoe, kind):
    """K = 4096: above an expert's index stands its start as the hash of its own first scales gives it, every place among them; under
    it, and everywhere else, both schedules write what the host mirror writes (the schedule kernel the launch constants too), and
    the mirror's decode functions read the device's records."""
    from expert_specialization_moe_amd import _native, workloads as W

    lib, n, k = _native.lib, 640, 4096
    rows = [(5, 64, 0, 70, 33, 200, 1, 16)[i % 8] for i in range(96)]
    experts, bits = len(rows), 1 if kind == "mx" else 0
    prob = W.Problem("starts", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands)(prob, "cuda", seed=9, out_dtype=torch.bfloat16, weight_std=0.05)
    scales = ops["sfb_phys" if kind == "mx" else "scales_b_phys"].reshape(experts, -1).contiguous().view(torch.uint8).cpu().numpy()
    starts = [H.k_start_blocks(scales[e].tobytes()) for e in range(experts)]
    assert set(starts) == {0, 4, 8, 12, 16, 20, 24, 28}
    words = lib.esmoe_gemm_workspace_bytes(experts) // 4
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    ps, host = np.array([[m, n, k] for m in rows], dtype=np.int32), np.zeros(words, dtype=np.int32)
    assert lib.esmoe_host_schedule(ptr(ps), experts, n, 0, bits, ptr(host)) == 0, _native.last_error()
    ws = torch.full((words,), -1, dtype=torch.int32, device="cuda").view(torch.uint8)
    out = torch.full_like(ops["output"], 3.0)
    _mm(_native, ops, kind, ws, out)
    own = _mm(_native, ops, kind, None, torch.full_like(out, 3.0))
    assert torch.equal(own.view(torch.int16), out.view(torch.int16))
    kernel, first = ws.view(torch.int32).cpu().numpy(), 64 + 32 * 8
    want = host[first:first + 4 * (experts + 1)].reshape(-1, 4).copy()
    want[:-1, 2] |= np.array([starts[e] // 4 for e in want[:-1, 2]], dtype=np.int32) << 16
    for dev in (kernel, _read_stream_workspace(_native, words)):
        got = dev[first:first + 4 * (experts + 1)].reshape(-1, 4)
        assert np.array_equal(got, want), np.flatnonzero((got != want).any(axis=1))
    header = [1, 2, 3, 4, 5, 16, 32] + [64 + 32 * x for x in range(8)]
    assert kernel[header].tolist() == host[header].tolist()
    tile, mirror = np.zeros(5, dtype=np.int32), np.zeros(5, dtype=np.int32)
    for item in range(int(host[1])):
        rc = [lib.esmoe_host_decode_light(ptr(ps), ptr(w), experts, n, 0, bits, item, ptr(t)) for w, t in ((kernel, tile), (host, mirror))]
        assert rc[0] == rc[1] and (rc[0] or np.array_equal(tile, mirror)), item
    for xcd in range(8):
        for ticket in range(64):
            rc = [lib.esmoe_host_decode_heavy(ptr(ps), ptr(w), experts, n, 0, bits, xcd, ticket, ptr(t)) for w, t in ((kernel, tile), (host, mirror))]
            assert rc[0] == rc[1] and (rc[0] or np.array_equal(tile, mirror)), (xcd, ticket)
