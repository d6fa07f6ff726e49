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
    from expert_specialization_moe_amd import _native, workloads as W

    rows, n, k = CASES[name]
    experts, total = len(rows), sum(rows)
    gen = torch.Generator(device="cuda").manual_seed(experts + n)
    ints = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device="cuda").float()
    a, b = ints(total + 1, k), ints(experts, n, k)   # (a spare row that belongs to no expert)
    bso, sf_rows = W.blockscale_offsets_of(rows)
    ops = dict(a=a.to(torch.float8_e4m3fn), b_phys=b.to(torch.float8_e4m3fn),
               problem_sizes=torch.tensor([[m, n, k] for m in rows], dtype=torch.int32, device="cuda"),
               expert_offsets=torch.tensor(W.offsets_of(rows), dtype=torch.int32, device="cuda"),
               blockscale_offsets=torch.tensor(bso, dtype=torch.int32, device="cuda"))
    if kind == "mx":   # unit scales
        ops["sfa"] = torch.full((max(int(sf_rows), 128), k // 32), 127, device="cuda", dtype=torch.uint8)
        ops["sfb_phys"] = torch.full((experts * n, k // 32), 127, device="cuda", dtype=torch.uint8)
    else:
        ops["scales_a"] = torch.ones((total + 1, k // 128), device="cuda")
        ops["scales_b_phys"] = torch.ones((experts, n // 128, k // 128), device="cuda")
    want = torch.full((total + 2, n), 3.0, dtype=torch.bfloat16, device="cuda")
    off = 0
    for i, m in enumerate(rows):
        want[off:off + m] = (a[off:off + m].double() @ b[i].double().t()).float().to(torch.bfloat16)
        off += m
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
