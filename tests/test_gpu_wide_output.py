"""Outputs so wide that the 64 rows of a short tile pass 2^30 and 2^32 bytes: stores must reach their element, and the absent
half of a last column tile of 128 columns must be dropped.  Small-integer operands make every sum exact, so every element
must equal the product rounded once."""
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("fp8", (1 << 23) + 128), ("mx", (1 << 23) + 128), ("fp8", (1 << 24) + 128), ("fp8", (1 << 25) + 128),
                                    ("mx", (1 << 25) + 256)])
def test_wide_output(esmoe, kind, n):
    from expert_specialization_moe_amd import _native

    k, rows = 128, 64
    gen = torch.Generator(device="cuda").manual_seed(n)
    a = torch.randint(-2, 3, (rows, k), generator=gen, device="cuda").to(torch.float8_e4m3fn)
    codes = torch.tensor([-2.0, -1.0, 0.0, 1.0, 2.0], device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
    b = torch.empty((1, n, k), dtype=torch.uint8, device="cuda")
    step = 1 << 20
    for n0 in range(0, n, step):
        part = b[0, n0:n0 + step]
        part.copy_(codes[torch.randint(0, 5, part.shape, generator=gen, device="cuda")])
    ops = dict(a=a, b_phys=b.view(torch.float8_e4m3fn), output=torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device="cuda"),
               problem_sizes=torch.tensor([[rows, n, k]], dtype=torch.int32, device="cuda"),
               expert_offsets=torch.zeros(1, dtype=torch.int32, device="cuda"))
    if kind == "fp8":
        ops["scales_a"] = torch.ones((rows, 1), device="cuda")
        ops["scales_b_phys"] = torch.ones((1, n // 128, 1), device="cuda")
        y = H.capi_fp8_mm(_native, ops)
    else:
        ops["sfa"] = torch.full((128, k // 32), 127, dtype=torch.uint8, device="cuda")   # 2^0
        ops["sfb_phys"] = torch.full((n, k // 32), 127, dtype=torch.uint8, device="cuda")
        ops["blockscale_offsets"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        y = H.capi_mx_mm(_native, ops)
    for n0 in range(0, n, step):
        want = a.float() @ ops["b_phys"][0, n0:n0 + step].float().t()
        assert torch.equal(y[:, n0:n0 + step].float(), want.to(torch.bfloat16).float()), f"columns from {n0}"
