"""K orders that start in the middle (K a multiple of 4096): what an expert's bytes may depend on.

A row's bytes are the same however many other rows its expert has (short tiles, 128- and 192-row tiles, every K loop), with the
schedule of the GEMM kernel and that of the schedule kernel (a caller's workspace; more experts than the kernel schedules
itself).  The eight experts begin at four places at least, which is checked against the hash of their scales; each is also compared
with the fp64 product: one rounding to bfloat16 (2^-8 of the value) plus K roundings of fp32 sums (K * 2^-24 of the magnitudes' sum).
"""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [4096, 8192])
@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_a_rows_bytes_do_not_depend_on_the_other_rows(esmoe, kind, k):
    from expert_specialization_moe_amd import _native, workloads as W

    n, experts, rows = 512, 8, 330
    prob = W.Problem("start", n, k, [rows] * experts, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    make = W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands
    ops = make(prob, "cuda", seed=k, out_dtype=torch.bfloat16, weight_std=0.05)
    scales = ops["sfb_phys" if kind == "mx" else "scales_b_phys"].reshape(experts, -1).contiguous().view(torch.uint8).cpu().numpy()
    starts = [H.k_start_blocks(scales[e].tobytes()) for e in range(experts)]
    assert len(set(starts)) >= 4 and any(starts), starts
    fresh = lambda: torch.full_like(ops["output"], 3.0)
    base = _mm(_native, ops, kind, None, fresh()).clone()
    offs = [e * rows for e in range(experts)]
    for sizes in ([1, 16, 17, 33, 64, 65, 129, 193], [200, 130, 70, 64, 40, 20, 5, 0]):
        less = dict(ops, problem_sizes=torch.tensor([[m, n, k] for m in sizes], dtype=torch.int32, device="cuda"))
        ws = torch.zeros((_native.lib.esmoe_gemm_workspace_bytes(experts),), dtype=torch.uint8, device="cuda")
        for workspace in (None, ws):
            got = _mm(_native, less, kind, workspace, fresh())
            for e, m in enumerate(sizes):
                lo = offs[e]
                assert torch.equal(got[lo:lo + m].view(torch.int16), base[lo:lo + m].view(torch.int16)), (e, m)
                assert (got[lo + m:lo + rows] == 3.0).all(), (e, m)
    if kind == "fp8":
        a = ops["a"].double() * ops["scales_a"].double().repeat_interleave(128, dim=1)
        sb = ops["scales_b_phys"].double().repeat_interleave(128, dim=1).repeat_interleave(128, dim=2)
        for e in range(experts):
            w, sl = ops["b_phys"][e].double() * sb[e], slice(offs[e], offs[e] + rows)
            ref, mag = a[sl] @ w.t(), a[sl].abs() @ w.abs().t()
            assert ((base[sl].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * (k * 2.0 ** -24)).all(), e


def test_more_experts_than_the_kernel_schedules_itself(esmoe):
    """520 experts through the schedule kernel against the same rows in two calls that the kernel schedules itself."""
    from expert_specialization_moe_amd import _native, workloads as W

    n, k, experts, m = 128, 4096, 520, 3
    rows = [m] * experts
    prob = W.Problem("many", n, k, rows)
    ops = W.make_fp8_blockwise_operands(prob, "cuda", seed=1, out_dtype=torch.bfloat16, weight_std=0.05)
    whole = _mm(_native, ops, "fp8", None, torch.full_like(ops["output"], 3.0)).clone()
    half = experts // 2
    for i in range(2):
        sl, rl = slice(i * half, (i + 1) * half), slice(i * half * m, (i + 1) * half * m)
        part = dict(a=ops["a"][rl].contiguous(), scales_a=ops["scales_a"][rl].contiguous(), b_phys=ops["b_phys"][sl].contiguous(),
                    scales_b_phys=ops["scales_b_phys"][sl].contiguous(), problem_sizes=ops["problem_sizes"][sl].contiguous(),
                    expert_offsets=(ops["expert_offsets"][sl] - i * half * m).contiguous())
        got = _mm(_native, part, "fp8", None, torch.full_like(ops["output"][rl], 3.0))
        assert torch.equal(got.view(torch.int16), whole[rl].view(torch.int16)), i


@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_scales_that_begin_four_bytes_behind_a_16_byte_boundary(esmoe, kind):
    """The entry points ask for four bytes: the same bytes as with aligned scales, in both schedules, short and tall tiles."""
    from expert_specialization_moe_amd import _native, workloads as W

    n, k, rows = 384, 4096, [5, 64, 0, 200, 33]
    prob = W.Problem("under", n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    make = W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands
    ops = make(prob, "cuda", seed=4, out_dtype=torch.bfloat16, weight_std=0.05)
    base = _mm(_native, ops, kind, None, torch.full_like(ops["output"], 3.0)).clone()
    moved = dict(ops)
    for name in ("sfa", "sfb_phys") if kind == "mx" else ("scales_a", "scales_b_phys"):
        buffer = torch.empty((4 + ops[name].numel() * ops[name].element_size(),), dtype=torch.uint8, device="cuda")
        moved[name] = buffer[4:].view(ops[name].dtype).view(ops[name].shape)
        moved[name].copy_(ops[name])
        assert moved[name].data_ptr() % 16 == 4
    ws = torch.zeros((_native.lib.esmoe_gemm_workspace_bytes(len(rows)),), dtype=torch.uint8, device="cuda")
    for workspace in (None, ws):
        got = _mm(_native, moved, kind, workspace, torch.full_like(base, 3.0))
        assert torch.equal(got.view(torch.int16), base.view(torch.int16))
