"""Launches whose queues hold runs (K > 512) on the GPU: 96- and 160-row tiles at their edges, and the hand-out around 256 and 512 heavy
tiles, both formats, plain and with the fused epilogues.  An output element's sums are in one order whatever tile it is in, so the bytes
have to be those of a forced tile height, which blocks hand out; the forced heights have their own tests against the oracle."""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm

pytestmark = pytest.mark.gpu

EDGES = [65, 80, 81, 96, 97, 128, 129, 144, 145, 160, 161, 192, 193, 208, 224, 225, 256, 257, 288, 289, 300, 352, 353, 64, 33, 0, 1]


@pytest.mark.parametrize("name,rows,n,k", [
    ("edges", EDGES, 640, 640), ("edges from the middle of K", EDGES, 512, 4096), ("edges", EDGES, 256, 2176), ("rows of blocks", [1700, 70, 3], 768, 768),
    ("255 tiles", [70] * 255, 256, 640), ("257 tiles", [100] * 257, 256, 640), ("513 tiles", [66] * 513, 256, 640)])
@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_same_bytes_as_a_forced_height(esmoe, kind, name, rows, n, k):
    from expert_specialization_moe_amd import _native
    from expert_specialization_moe_amd import workloads as W

    print(kind, name, flush=True)
    prob = W.Problem(name, n, k, rows, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands)(prob, "cuda", seed=3, weight_std=0.05)
    want = _mm(_native, ops, kind, None, torch.full_like(ops["output"], float("nan")), 64).clone()
    assert not torch.isnan(want).any()
    ws = torch.zeros((_native.lib.esmoe_gemm_workspace_bytes(len(rows)),), dtype=torch.uint8, device="cuda")
    for workspace in (None, ws, None):
        got = _mm(_native, ops, kind, workspace, torch.full_like(ops["output"], float("nan")))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("kind", ["fp8", "mx"])
def test_fused_epilogues_of_the_new_heights(esmoe, kind):
    """Bytes and scales of the projection followed by the stand-alone SwiGLU quantiser; MXFP8: also the zero scale bytes of padding rows."""
    from expert_specialization_moe_amd import ops as P
    from expert_specialization_moe_amd import workloads as W

    n, k, e, total = 512, 640, len(EDGES), sum(EDGES)
    prob = W.Problem("fused", n, k, EDGES, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands)(prob, "cuda", seed=4, weight_std=0.05)
    q = [torch.full((total, n // 2), 1.0, device="cuda").to(torch.float8_e4m3fn) for _ in range(2)]
    if kind == "fp8":
        s = [torch.full((total, n // 256), -1.0, device="cuda") for _ in range(2)]
        P.es_fp8_blockwise_scaled_grouped_mm(ops["output"], ops["a"], ops["b"], ops["scales_a"], ops["scales_b"], ops["stride_a"], ops["stride_b"],
                                             ops["stride_d"], ops["problem_sizes"], ops["expert_offsets"], ops["workspace"])
        P.es_swiglu_quant_1x128(ops["output"], q[0], s[0])
        P.es_fp8_blockwise_scaled_grouped_mm_swiglu_quant(q[1], s[1], ops["a"], ops["b"], ops["scales_a"], ops["scales_b"], ops["problem_sizes"],
                                                          ops["expert_offsets"], ops["workspace"], ops["output"].dtype)
    else:
        sf_rows = W.blockscale_offsets_of(EDGES)[1]
        s = [torch.full((int(sf_rows), n // 64), 7, dtype=torch.uint8, device="cuda") for _ in range(2)]
        meta = (ops["problem_sizes"], ops["expert_offsets"], ops["blockscale_offsets"])
        P.es_sm100_mxfp8_blockscaled_grouped_mm(ops["output"], ops["a"], ops["b"], ops["sfa"], ops["sfb"], *meta)
        P.es_swiglu_mxfp8_grouped_quant(ops["output"], *meta, q[0], s[0])
        P.es_mxfp8_blockscaled_grouped_mm_swiglu_quant(q[1], s[1], ops["a"], ops["b"], ops["sfa"], ops["sfb"], *meta, ops["output"].dtype)
    torch.cuda.synchronize()
    assert torch.equal(q[0].view(torch.uint8), q[1].view(torch.uint8)) and torch.equal(s[0], s[1])
