"""Half items of fused MXFP8 launches on the GPU where an expert's K order starts in the middle (K a multiple of 4096), with the shortest K
that has them, behind whole items and behind tall tiles; both output types.  Bit-exact against the projection and the quantiser by themselves."""
import pytest
import torch

from tests.test_gpu_mx_fused_swiglu import _fused, _separate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,inter,k,rows", [
    ("one round", 256, 256, [1, 16, 17, 32, 33, 64, 0, 50]), ("one round", 384, 4096, [64, 1, 16, 17, 0, 33, 20]),
    ("long K", 128, 5504, [7, 40, 64]), ("behind whole items", 128, 1024, [1 + i % 64 for i in range(270)]),
    ("behind tall tiles", 512, 4096, [100, 70, 200, 90] * 16 + [9, 64, 33])])
def test_bytes_of_the_separate_route(esmoe, name, inter, k, rows, dtype):
    from expert_specialization_moe_amd import _native
    from expert_specialization_moe_amd import workloads as W

    print(name, inter, k, dtype, flush=True)
    prob = W.Problem("gate_up", 2 * inter, k, rows)
    ops = W.make_mxfp8_operands(prob, "cuda", seed=5, out_dtype=dtype, weight_std=0.05)
    q, sf = _fused(_native, ops, rows, inter, dtype)
    q_ref, sf_ref = _separate(esmoe, _native, ops, rows, inter, dtype, 0)
    assert torch.equal(q, q_ref), f"{(q != q_ref).sum().item()} bytes differ"
    assert torch.equal(sf, sf_ref), f"{(sf != sf_ref).sum().item()} scale bytes differ"
