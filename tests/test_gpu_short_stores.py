"""Output stores of the short tiles: 16 bytes a lane from two column tiles (whole tiles) or two row tiles (halves of 128 columns),
with and without the non-temporal hint.

240 items, of which the last 128 go out as halves; every tile height with full and ragged rows, K around the places where the
hint changes (4 and 12 K blocks, 8 rows), both output types, a last column tile of 128.  Small-integer operands make every sum
exact: the output must equal the fp64 product rounded once, and rows behind the last expert's stay as they were.  An output that
begins 8 bytes behind a 16-byte boundary, the least that the entry points ask for, gets the same.
"""
import pytest
import torch

from tests import helpers as H
from tests.test_gpu_one_launch import _mm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kblocks", [1, 3, 4, 11, 12, 13])
def test_short_tiles_store_every_element_once(esmoe, kblocks, dtype):
    from expert_specialization_moe_amd import _native, workloads as W

    rows = [(1, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 0)[i % 12] for i in range(88)]
    experts, total, n, k, spare = len(rows), sum(rows), 640, kblocks * 128, 3
    gen = torch.Generator(device="cuda").manual_seed(k)
    ints = lambda *shape: torch.randint(-2, 3, shape, generator=gen, device="cuda").float()
    a, b = ints(total, k), ints(experts, n, k)
    ops = dict(a=a.to(torch.float8_e4m3fn), b_phys=b.to(torch.float8_e4m3fn),
               scales_a=torch.exp2(ints(total, kblocks)), scales_b_phys=torch.exp2(ints(experts, n // 128, kblocks)),
               problem_sizes=torch.tensor([[m, n, k] for m in rows], dtype=torch.int32, device="cuda"),
               expert_offsets=torch.tensor(W.offsets_of(rows), dtype=torch.int32, device="cuda"))
    want = torch.full((total + spare, n), 3.0, dtype=dtype, device="cuda")
    off = 0
    for i, m in enumerate(rows):
        ai = a[off:off + m].double() * ops["scales_a"][off:off + m].double().repeat_interleave(128, dim=1)
        bi = b[i].double() * ops["scales_b_phys"][i].double().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)
        want[off:off + m] = (ai @ bi.t()).float().to(dtype)
        off += m
    for front in (0, 4):
        buffer = torch.full((front + want.numel(),), 3.0, dtype=dtype, device="cuda")
        got = buffer[front:].view(want.shape)
        assert got.data_ptr() % 16 == 2 * front
        _mm(_native, ops, "fp8", None, got[:total])
        assert torch.equal(got.contiguous().view(torch.int16), want.view(torch.int16)), front
        assert (buffer[:front] == 3.0).all()
