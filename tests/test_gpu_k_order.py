"""One K order for every tile and every place in the list, also where rows are a multiple of 4096 bytes apart.

Every output element is accumulated K block by K block in one order that is the expert's own (from the first block to the last or,
for K a multiple of 4096, from a place that the expert's first weight scales give, and round), whatever tile computes it and wherever its
expert stands in the call: every forced tile height must give the bytes of the device schedule, the fused epilogues those of
projection -> stand-alone quantiser, and an expert listed elsewhere, or in a call of its own, its own bytes again (another
rank's share of the same experts is such a call).  FP8-blockwise is also checked against
a product of the dequantised operands in fp64: one rounding to bfloat16 (2^-8 of the value) plus K roundings of fp32 sums
(K * 2^-24 of the sum of the products' magnitudes).  MXFP8 against the same with the oracle's dequantisation and a tighter
count: a sum passes one MFMA of 128 products and one addition per K block, K / 128 + 128 steps that lose at most 2^-23 of
the magnitudes' sum each (whether they round or cut off).
"""
import numpy as np
import pytest
import torch

from oracle import mxfp8 as omx
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4096, 8192, 12288])
@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_wrapped_k_order_is_the_same_for_every_tile(esmoe, kind, k):
    from expert_specialization_moe_amd import _native, workloads as W

    n, rows = 512, [1, 200, 0, 33, 16, 130, 64, 65, 400, 7, 17]   # every tile height and its edges
    dt = torch.bfloat16
    prob = W.Problem("wrap", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    if kind == "mx":
        ops = W.make_mxfp8_operands(prob, "cuda", seed=k, out_dtype=dt, weight_std=0.05)
        mm = H.capi_mx_mm
    else:
        ops = W.make_fp8_blockwise_operands(prob, "cuda", seed=k, out_dtype=dt, weight_std=0.05)
        mm = H.capi_fp8_mm
    base = mm(_native, ops, 0, out=torch.full_like(ops["output"], 3.0)).clone()
    for bm in (16, 32, 64, 128, 192):
        forced = mm(_native, ops, bm, out=torch.full_like(ops["output"], 3.0))
        assert torch.equal(base.view(torch.int16), forced.view(torch.int16)), f"tile height {bm}"
    if kind == "fp8":
        a = ops["a"].double() * ops["scales_a"].double().repeat_interleave(128, dim=1)
        sb = ops["scales_b_phys"].double().repeat_interleave(128, dim=1).repeat_interleave(128, dim=2)
        off = 0
        for i, m in enumerate(rows):
            w = ops["b_phys"][i].double() * sb[i]
            ref, mag = a[off:off + m] @ w.t(), a[off:off + m].abs() @ w.abs().t()
            bound = ref.abs() * 2.0 ** -8 + mag * (k * 2.0 ** -24)
            assert ((base[off:off + m].double() - ref).abs() <= bound).all(), f"expert {i}"
            off += m
        q = torch.zeros((off, n // 2), dtype=torch.uint8, device="cuda")
        sc = torch.zeros((off, n // 256), dtype=torch.float32, device="cuda")
        esmoe.es_fp8_blockwise_scaled_grouped_mm_swiglu_quant(q, sc, ops["a"], ops["b"], ops["scales_a"], ops["scales_b"],
                                                              ops["problem_sizes"], ops["expert_offsets"], ops["workspace"], dt)
        q2, sc2 = esmoe.es_swiglu_quant_1x128(base)
        assert torch.equal(q, q2.view(torch.uint8)) and torch.equal(sc, sc2)
    else:
        codes, scales = H.codes(ops["a"]), omx.unswizzle_scales
        off = 0
        for i, m in enumerate(rows):
            if m:
                sa = scales(ops["sfa"].cpu().numpy().reshape(-1), m, k, base=int(ops["blockscale_offsets"][i]) * (k // 32))
                sw = scales(ops["sfb_phys"].cpu().numpy().reshape(-1), n, k, base=i * n * (k // 32))
                a, w = omx.dequant_rows(codes[off:off + m], sa).astype(np.float64), omx.dequant_rows(H.codes(ops["b_phys"][i]), sw).astype(np.float64)
                ref, mag = a @ w.T, np.abs(a) @ np.abs(w).T
                y = H.f32(base[off:off + m]).astype(np.float64)
                bound = np.abs(ref) * 2.0 ** -8 + mag * ((k / 128 + 128) * 2.0 ** -23)
                assert (np.abs(y - ref) <= bound).all(), f"expert {i}"
            off += m
        q = torch.zeros((sum(rows), n // 2), dtype=torch.uint8, device="cuda")
        sf = torch.zeros((ops["sfa"].shape[0], n // 64), dtype=torch.uint8, device="cuda")
        esmoe.es_mxfp8_blockscaled_grouped_mm_swiglu_quant(q, sf, ops["a"], ops["b"], ops["sfa"], ops["sfb"], ops["problem_sizes"],
                                                           ops["expert_offsets"], ops["blockscale_offsets"], dt)
        q2, sf2 = torch.zeros_like(q), torch.zeros_like(sf)
        esmoe.es_swiglu_mxfp8_grouped_quant(base, ops["problem_sizes"], ops["expert_offsets"], ops["blockscale_offsets"], q2, sf2)
        assert torch.equal(q, q2) and torch.equal(sf, sf2)


@pytest.mark.parametrize("k", [4096, 8192, 12288, 7168])
@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_an_experts_bytes_do_not_depend_on_its_place_in_the_list(esmoe, kind, k):
    from expert_specialization_moe_amd import _native, workloads as W

    n, rows = 512, [1, 200, 0, 33, 16, 130, 64, 400, 7]
    prob = W.Problem("place", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    make, mm = (W.make_mxfp8_operands, H.capi_mx_mm) if kind == "mx" else (W.make_fp8_blockwise_operands, H.capi_fp8_mm)
    ops = make(prob, "cuda", seed=k, out_dtype=torch.bfloat16, weight_std=0.05)
    base = mm(_native, ops, 0).clone()
    offs = W.offsets_of(rows)
    weights = ("b_phys", "sfb_phys") if kind == "mx" else ("b_phys", "scales_b_phys")
    lists = [[8, 7, 6, 5, 4, 3, 2, 1, 0], [3, 0, 8, 1, 7, 2, 6, 4, 5]] + [[e] for e in range(len(rows))]
    for order in lists:
        moved = dict(ops, output=torch.full_like(ops["output"], float("nan")))
        for name in weights + ("problem_sizes", "expert_offsets") + (("blockscale_offsets",) if kind == "mx" else ()):
            moved[name] = (ops[name].view(len(rows), n, k // 32) if name == "sfb_phys" else ops[name])[order].contiguous()
        got = mm(_native, moved, 0)
        for e in order:
            sl = slice(int(offs[e]), int(offs[e]) + rows[e])
            assert torch.equal(got[sl].view(torch.int16), base[sl].view(torch.int16)), f"expert {e} of {order}"


@pytest.mark.parametrize("k", [4096, 7168])
@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_columns_of_an_expert_by_themselves(esmoe, kind, k):
    """The first columns give the bytes they have in the whole, whatever K; later ones too unless K is a multiple of 4096, where they are
    the same sums in another order: both results lie within K roundings of fp32 sums (K * 2^-24 of the magnitudes' sum) and
    one rounding to bfloat16 (2^-8) of the exact value."""
    from expert_specialization_moe_amd import _native, workloads as W

    n, rows = 768, [1, 200, 0, 33, 130, 64]
    experts = len(rows)
    prob = W.Problem("columns", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    make, mm = (W.make_mxfp8_operands, H.capi_mx_mm) if kind == "mx" else (W.make_fp8_blockwise_operands, H.capi_fp8_mm)
    ops = make(prob, "cuda", seed=k + 1, out_dtype=torch.bfloat16, weight_std=0.05)
    whole = mm(_native, ops, 0, out=torch.full_like(ops["output"], 3.0)).clone()
    for lo, hi in ((0, 128), (0, 384), (256, 768), (384, 512)):
        part = dict(ops, b_phys=ops["b_phys"][:, lo:hi].contiguous())
        if kind == "mx":
            part["sfb_phys"] = ops["sfb_phys"].view(experts, n, k // 32)[:, lo:hi].contiguous()
        else:
            part["scales_b_phys"] = ops["scales_b_phys"][:, lo // 128:hi // 128].contiguous()
        part["problem_sizes"] = torch.tensor([[m, hi - lo, k] for m in rows], dtype=torch.int32, device="cuda")
        want = whole[:, lo:hi].contiguous()
        got = mm(_native, part, 0, out=torch.full_like(want, 3.0))
        if lo == 0 or k % 4096:
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (lo, hi)
        elif kind == "fp8":
            a = ops["a"].double() * ops["scales_a"].double().repeat_interleave(128, dim=1)
            off = 0
            for e, m in enumerate(rows):
                w = part["b_phys"][e].double() * part["scales_b_phys"][e].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
                mag = a[off:off + m].abs() @ w.abs().t()
                diff = (got[off:off + m].double() - want[off:off + m].double()).abs()
                assert (diff <= 2 * (want[off:off + m].double().abs() * 2.0 ** -8 + mag * (k * 2.0 ** -24))).all(), (lo, hi, e)
                off += m
