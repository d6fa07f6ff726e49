"""The fused epilogues behind tall tiles of every height where an expert's K order starts in the middle and wraps (K a multiple of 4096) and
with a K of 43 blocks, both formats and output types.  Bytes and scales of the projection followed by the SwiGLU quantiser."""
import pytest
import torch

from tests.test_gpu_runs import EDGES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,k,dtype", [("fp8", 4096, torch.bfloat16), ("fp8", 4096, torch.float16), ("fp8", 5504, torch.bfloat16),
                                          ("mx", 4096, torch.bfloat16), ("mx", 4096, torch.float16), ("mx", 5504, torch.float16)])
def test_bytes_of_the_projection_and_the_quantiser(esmoe, kind, k, dtype):
    from expert_specialization_moe_amd import ops as P
    from expert_specialization_moe_amd import workloads as W

    print(kind, k, dtype, flush=True)
    n, total = 512, sum(EDGES)
    prob = W.Problem("fused", n, k, EDGES, kind="mxfp8" if kind == "mx" else "fp8_blockwise")
    ops = (W.make_mxfp8_operands if kind == "mx" else W.make_fp8_blockwise_operands)(prob, "cuda", seed=6, out_dtype=dtype, weight_std=0.05)
    assert ops["output"].dtype == dtype
    q = [torch.full((total, n // 2), 1.0, device="cuda").to(torch.float8_e4m3fn) for _ in range(2)]
    if kind == "fp8":
        s = [torch.full((total, n // 256), -1.0, device="cuda") for _ in range(2)]
        P.es_fp8_blockwise_scaled_grouped_mm(ops["output"], ops["a"], ops["b"], ops["scales_a"], ops["scales_b"], ops["stride_a"], ops["stride_b"],
                                             ops["stride_d"], ops["problem_sizes"], ops["expert_offsets"], ops["workspace"])
        P.es_swiglu_quant_1x128(ops["output"], q[0], s[0])
        P.es_fp8_blockwise_scaled_grouped_mm_swiglu_quant(q[1], s[1], ops["a"], ops["b"], ops["scales_a"], ops["scales_b"], ops["problem_sizes"],
                                                          ops["expert_offsets"], ops["workspace"], dtype)
    else:
        s = [torch.full((int(W.blockscale_offsets_of(EDGES)[1]), n // 64), 7, dtype=torch.uint8, device="cuda") for _ in range(2)]
        meta = (ops["problem_sizes"], ops["expert_offsets"], ops["blockscale_offsets"])
        P.es_sm100_mxfp8_blockscaled_grouped_mm(ops["output"], ops["a"], ops["b"], ops["sfa"], ops["sfb"], *meta)
        P.es_swiglu_mxfp8_grouped_quant(ops["output"], *meta, q[0], s[0])
        P.es_mxfp8_blockscaled_grouped_mm_swiglu_quant(q[1], s[1], ops["a"], ops["b"], ops["sfa"], ops["sfb"], *meta, dtype)
    torch.cuda.synchronize()
    assert q[0].float().abs().max() > 1
    assert torch.equal(q[0].view(torch.uint8), q[1].view(torch.uint8)) and torch.equal(s[0], s[1])
