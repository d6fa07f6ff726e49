"""Strips: light tickets drawn together that are neighbouring column tiles of one expert run as one stream of stages.

Many short items per workgroup, so that the first draws take several tickets each: strips of 2 up to more tiles than an
expert has (a draw then crosses experts), cut at the last column tile of 128 columns and in front of the narrow tail.  The
forced 64-row height walks the same tiles one by one, so its bytes must be equal; small-integer operands make every sum
exact, so the result must also equal the fp64 product rounded once.  Rows past an expert's last must not be written.
"""
import pytest
import torch

from tests import helpers as H

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
    # the library's workspace (one launch), the path of the public operators
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
