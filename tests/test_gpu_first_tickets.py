"""First tickets: a workgroup's first ticket goes by its index, the counters hand out the rest, and a launch of first tickets
only uses no counter.

The row lists sit at the edges: launches with fewer tickets than workgroups, as many, one more; heavy queues of no, one and two
blocks; both kinds; nothing at all.  Small-integer operands make every sum exact, so the output must equal the fp64 product
rounded once; the library's workspace must hold zero counters after every call.
"""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm, _read_stream_workspace

pytestmark = pytest.mark.gpu

CASES = {
    "nothing": ([0, 0, 0], 512, 512),
    "one_ticket": ([0, 5], 128, 256),
    "under_a_ticket_each": ([8] * 60, 512, 256),
    "a_ticket_each": ([9] * 64, 512, 384),            # 64 items of 256 columns, handed out as 128 halves; x 2 = 256 tickets
    "one_more": ([9] * 64 + [1], 512, 384),
    "two_draws": ([3] * 400, 512, 128),
    "one_heavy_block": ([200, 0], 1024, 256),
    "a_block_a_queue": ([100] * 8, 512, 256),
    "nine_blocks": ([100] * 9, 512, 256),
    "both": ([100] * 5 + [7] * 30, 768, 512),
    "many_of_both": ([70] * 20 + [16] * 300 + [400], 384, 256),
    "blocks_of_three": ([150] * 70, 768, 256),       # 9 a queue; four tickets of each of the first eight are first ones
    "blocks_of_one": ([65] * 300, 256, 128),
    "blocks_of_sixteen": ([1500] * 17, 512, 128),
    "blocks_of_eighteen": ([1100] * 9, 640, 128),     # handed out as blocks of 32
    "small_blocks_and_light": ([100] * 40 + [3] * 60, 512, 256),
}


@pytest.mark.parametrize("kind", ["fp8", "mx"])
@pytest.mark.parametrize("name", list(CASES))
def test_calls_at_the_edges_of_the_first_tickets(esmoe, kind, name):
    from expert_specialization_moe_amd import _native

    rows, n, k = CASES[name]
    experts, total = len(rows), sum(rows)
    ops, product = H.integer_operands(kind, rows, n, k, experts + n, spare=1)   # (a spare row that belongs to no expert)
    want = torch.full((total + 2, n), 3.0, dtype=torch.bfloat16, device="cuda")
    want[:total] = product.float().to(torch.bfloat16)
    for rep in range(2):
        got = torch.full_like(want, 3.0)
        _mm(_native, ops, kind, None, got[:total + 1])
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), rep
        counters = _read_stream_workspace(_native, 64 + 32 * 8)[[16, 32] + [64 + 32 * x for x in range(8)]]
        assert not counters.any(), counters
    ws = torch.randint(0, 256, (_native.lib.esmoe_gemm_workspace_bytes(experts),), dtype=torch.uint8, device="cuda")
    got = torch.full_like(want, 3.0)
    _mm(_native, ops, kind, ws, got[:total + 1])
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
