"""Heavy tickets that are no tiles: a block has 32 tickets whatever its size, and the queue moves on to its next block as soon as
one behind the block's last tile is drawn.

Blocks of one row and few columns (most tickets are none), a last row of blocks that is lower than the others, a last column of
blocks that is narrower, one to many blocks a queue, with and without light experts beside them.  Small-integer operands make
every sum exact; calls in a row on the library's workspace, whose counters must be zero after each.
"""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm, _read_stream_workspace

pytestmark = pytest.mark.gpu

CASES = {
    "one_by_three": ([100] * 90, 640), "two_by_five": ([200] * 70, 1280), "five_and_four_rows": ([1700, 1650, 1600], 1536),
    "narrow_last_column": ([700, 90, 300], 256 * 13), "one_tile_blocks": ([65] * 40, 256), "with_light": ([100] * 30 + [5, 0, 64, 33] * 40, 768),
    "few": ([400, 66], 384),
}


@pytest.mark.parametrize("kind", ["fp8", "mx"])
@pytest.mark.parametrize("name", list(CASES))
def test_every_tile_of_every_block_is_computed(esmoe, kind, name):
    from expert_specialization_moe_amd import _native

    rows, n = CASES[name]
    k, experts, total = 256, len(rows), sum(rows)
    ops, product = H.integer_operands(kind, rows, n, k, n + experts)
    want = torch.full((total + 1, n), 3.0, dtype=torch.bfloat16, device="cuda")
    want[:total] = product.float().to(torch.bfloat16)
    ws = torch.randint(0, 256, (_native.lib.esmoe_gemm_workspace_bytes(experts),), dtype=torch.uint8, device="cuda")
    for workspace in (None, None, ws):
        got = torch.full_like(want, 3.0)
        _mm(_native, ops, kind, workspace, got[:total])
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        counters = _read_stream_workspace(_native, 64 + 32 * 8)[[16, 32] + [64 + 32 * x for x in range(8)]]
        assert not counters.any(), counters
