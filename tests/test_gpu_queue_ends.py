"""Launches whose workgroups find heavy queues empty and look at all of them: queues of blocks with tickets that are no tiles (K <= 512) and
of runs, with and without light items, with every one of the three schedules (one wavefront's, the workgroup's, the schedule kernel's).
The bytes are those of a forced tile height, several calls in a row, and the counters are zero again."""
import pytest
import torch

from tests.test_gpu_one_launch import _mm, _read_stream_workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["fp8", "mx"])
@pytest.mark.parametrize("name,rows,n,k", [
    ("blocks of one queue more", [300, 70, 5, 200, 64] * 5, 1280, 256), ("blocks of 12 tiles", [250] * 40, 1536, 256), ("blocks, 100 experts", [90, 17, 0, 260] * 25, 768, 384),
    ("blocks, 600 experts", [70, 3] * 300, 256, 128), ("runs", [260, 8, 130] * 20, 1280, 640), ("runs, 600 experts", [66, 2] * 300, 256, 640),
    ("one queue", [193], 256, 256)])
def test_every_tile_once(esmoe, kind, name, rows, n, k):
    from expert_specialization_moe_amd import _native
    from expert_specialization_moe_amd import workloads as W

    print(kind, name, flush=True)
    prob = W.Problem(name, n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands)(prob, "cuda", seed=9, weight_std=0.05)
    want = _mm(_native, ops, kind, None, torch.full_like(ops["output"], float("nan")), 64).clone()
    assert not torch.isnan(want).any()
    ws = torch.zeros((_native.lib.esmoe_gemm_workspace_bytes(len(rows)),), dtype=torch.uint8, device="cuda")
    for workspace in (None, ws, None, None):
        got = _mm(_native, ops, kind, workspace, torch.full_like(ops["output"], float("nan")))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    dev = _read_stream_workspace(_native, 64 + 32 * 8)
    assert not dev[[16, 32] + [64 + 32 * x for x in range(8)]].any()
