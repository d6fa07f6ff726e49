"""Strips: light tickets drawn together that are neighbouring column tiles of one expert run as one stream of stages.

Many short items per workgroup, so that the first draws take several tickets each, with columns that end on a tile of 128.
The forced 64-row height walks the same tiles one by one, so its bytes must be equal; small-integer operands make every sum
exact, so the result must also equal the fp64 product rounded once.  Rows past an expert's last must not be written.
test_strips_give_the_bytes_of_single_tiles draws 1 to 4 tickets (on 256 CUs) on a caller's workspace; test_long_strips up to
32, whole experts and tickets of several experts, on the library's workspace, which is how the public operators call.
"""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm
from tests.test_strips_host import light_tickets, schedule_functions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,k,experts", [("fp8", 3200, 128, 200), ("fp8", 4096, 256, 96), ("fp8", 2176, 384, 160), ("fp8", 8192, 512, 70),
                                              ("fp8", 2048, 1536, 150), ("fp8", 1024, 4096, 300), ("mx", 3200, 128, 200), ("mx", 4096, 256, 96),
                                              ("mx", 2176, 640, 160), ("mx", 2048, 1024, 150)])
def test_strips_give_the_bytes_of_single_tiles(esmoe, kind, n, k, experts):
    from expert_specialization_moe_amd import _native, workloads as W

    rows = [(1, 0, 16, 17, 33, 64, 5, 32)[i % 8] for i in range(experts)]
    prob = W.Problem("strip", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    make = W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands
    ops = make(prob, "cuda", seed=k, out_dtype=torch.bfloat16, weight_std=0.05)
    spare = 3   # rows behind the last expert's, in the same buffer
    total = prob.total_rows
    big = torch.full((total + spare, n), 3.0, dtype=torch.bfloat16, device="cuda")
    mm = H.capi_mx_mm if kind == "mx" else H.capi_fp8_mm
    want = mm(_native, ops, 64, out=torch.zeros_like(ops["output"])).clone()
    # (a caller's workspace: a schedule kernel, then the GEMM kernel)
    if kind == "fp8":
        codes = torch.randint(-2, 3, (total, k), device="cuda").float()
        wcodes = torch.randint(-2, 3, (experts, n, k), device="cuda").float()
        exact = dict(ops, a=codes.to(torch.float8_e4m3fn), b_phys=wcodes.to(torch.float8_e4m3fn),
                     scales_a=torch.exp2(torch.randint(-2, 3, ops["scales_a"].shape, device="cuda").float()),
                     scales_b_phys=torch.exp2(torch.randint(-2, 3, ops["scales_b_phys"].shape, device="cuda").float()))
        y = mm(_native, exact, 0, out=torch.full_like(ops["output"], 3.0))
        off = 0
        for i, m in enumerate(rows):
            a = codes[off:off + m].double() * exact["scales_a"][off:off + m].double().repeat_interleave(128, dim=1)
            b = wcodes[i].double() * exact["scales_b_phys"][i].double().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)
            assert torch.equal(y[off:off + m], (a @ b.t()).float().to(torch.bfloat16)), f"expert {i}"
            off += m
    for rep in range(3):
        big.fill_(3.0)
        got = mm(_native, ops, 0, out=big[:total])
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), rep
        assert (big[total:] == 3.0).all()


@pytest.mark.parametrize("kind,n,k,experts,draw", [
    ("fp8", 7168, 256, 256, 14), ("mx", 7168, 256, 256, 14),   # half an expert's columns, K = 256
    ("fp8", 16384, 128, 260, 32), ("mx", 16384, 128, 260, 32),   # the longest there are: 32 tiles of one K block
    ("fp8", 4224, 128, 512, 17),       # all 17 column tiles of an expert, the last of 128 columns: draws cross experts
    ("fp8", 384, 128, 1024, 4), ("mx", 384, 128, 1024, 4),       # several experts in every draw (more than the library schedules itself)
    ("fp8", 1536, 512, 500, 6),           # a whole expert, K = 512
])
def test_long_strips(esmoe, tmp_path, kind, n, k, experts, draw):
    from expert_specialization_moe_amd import _native, workloads as W

    mx = kind == "mx"
    rows = [(1, 16, 17, 33, 64, 5, 32, 2)[(i * 5) % 8] for i in range(experts)]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    total_tickets, _, _ = light_tickets(_native, rows, n, 1 if mx else 0)
    if cus == 256:
        assert schedule_functions(tmp_path).draw(total_tickets, 0, cus, k // 128, 1) == draw
    gen = torch.Generator(device="cuda").manual_seed(n + experts)
    total, spare = sum(rows), 3
    ints = torch.tensor([-2.0, -1.0, 0.0, 1.0, 2.0], device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
    pick = lambda *shape: ints[torch.randint(0, 5, shape, generator=gen, device="cuda", dtype=torch.uint8).int()].view(torch.float8_e4m3fn)
    bso, sf_rows = W.blockscale_offsets_of(rows)
    ops = dict(a=pick(total, k), b_phys=pick(experts, n, k), problem_sizes=torch.tensor([[m, n, k] for m in rows], dtype=torch.int32, device="cuda"),
               expert_offsets=torch.tensor(W.offsets_of(rows), dtype=torch.int32, device="cuda"),
               blockscale_offsets=torch.tensor(bso, dtype=torch.int32, device="cuda"))
    if mx:   # any power of two per 32 values: products of one size range stay exact in fp32
        ops["sfa"] = torch.randint(125, 130, (int(sf_rows), k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        ops["sfb_phys"] = torch.randint(125, 130, (experts * n, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
    else:
        ops["scales_a"] = torch.exp2(torch.randint(-2, 3, (total, k // 128), generator=gen, device="cuda").float())
        ops["scales_b_phys"] = torch.exp2(torch.randint(-2, 3, (experts, n // 128, k // 128), generator=gen, device="cuda").float())
    fresh = lambda: torch.full((total + spare, n), 3.0, dtype=torch.bfloat16, device="cuda")
    single = fresh()
    _mm(_native, ops, kind, None, single[:total], 64)
    for rep in range(2):
        got = fresh()
        _mm(_native, ops, kind, None, got[:total])
        assert torch.equal(got.view(torch.int16), single.view(torch.int16)), rep
    assert (got[total:] == 3.0).all()
    if not mx:
        off = 0
        for i, m in enumerate(rows):
            a = ops["a"][off:off + m].double() * ops["scales_a"][off:off + m].double().repeat_interleave(128, dim=1)
            b = ops["b_phys"][i].double() * ops["scales_b_phys"][i].double().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)
            assert torch.equal(got[off:off + m], (a @ b.t()).float().to(torch.bfloat16)), f"expert {i}"
            off += m
