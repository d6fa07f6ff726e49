"""GPU parity of the routing metadata builder and the row packer: integers bit-exact against the oracle,
through the C ABI; then the whole caller-side chain on the device feeding the FP8 grouped GEMM."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import fp8_blockwise as ofp8
from oracle import routing as oroute
from tests import helpers as H

pytestmark = pytest.mark.gpu


def _capi_route(native, ids, first, experts, n, k, in_place=False):
    lib = native.lib
    pairs = ids.size
    d_ids = torch.from_numpy(ids.reshape(-1)).cuda()
    ps = torch.full((experts, 3), -7, dtype=torch.int32, device="cuda")
    eo = torch.full((experts + 1,), -7, dtype=torch.int32, device="cuda")
    bso = torch.full((experts + 1,), -7, dtype=torch.int32, device="cuda")
    dst = d_ids if in_place else torch.full((max(pairs, 1),), -7, dtype=torch.int32, device="cuda")
    wsb = lib.esmoe_route_workspace_bytes(pairs, experts)
    ws = torch.empty((wsb,), dtype=torch.uint8, device="cuda")
    rc = lib.esmoe_route_metadata(H.ptr(d_ids) if pairs else None, pairs, first, experts, n, k, H.ptr(ps), H.ptr(eo), H.ptr(bso),
                                  H.ptr(dst) if pairs else None, H.ptr(ws), wsb, H.stream_ptr())
    assert rc == 0, native.last_error()
    torch.cuda.synchronize()
    return ps.cpu().numpy(), eo.cpu().numpy(), bso.cpu().numpy(), dst.cpu().numpy()[:pairs]


@pytest.mark.parametrize("seed,pairs,experts,first,span", [(0, 0, 4, 0, 4), (1, 1, 1, 0, 1), (2, 777, 8, 16, 40), (3, 1024, 32, 0, 32),
                                                            (4, 1025, 32, 0, 256), (5, 32768, 32, 64, 256),
                                                            (6, 131072, 128, 0, 128), (7, 5000, 1024, 0, 1024),
                                                            (8, 4096, 3, 5, 6), (9, 16384, 256, 0, 300), (10, 16385, 256, 0, 300),
                                                            (11, 6579, 32, 0, 256), (12, 16384, 257, 0, 257)])
def test_route_metadata_bit_exact(esmoe, seed, pairs, experts, first, span):
    from expert_specialization_moe_amd import _native

    rng = np.random.default_rng(seed)
    ids = rng.integers(0, span, size=pairs).astype(np.int32)
    if pairs > 100:
        ids[:70] = first            # a long run of one expert inside one wavefront step
    got = _capi_route(_native, ids, first, experts, 4096, 7168)
    ref = oroute.route_metadata(ids, first, experts, 4096, 7168)
    for name, g, r in zip(("problem_sizes", "expert_offsets", "blockscale_offsets", "dst_row"), got, ref):
        assert np.array_equal(g, r), name


@pytest.mark.parametrize("pairs,experts,first,span", [(63, 2, 0, 2), (1023, 1023, 0, 1024), (2048, 64, 1, 64), (8192, 1024, 7, 2000),
                                                       (8193, 1024, 0, 1024), (16385, 1, 0, 3), (262144, 60, 0, 64),
                                                       (262145, 256, 0, 256), (600001, 100, 3, 128)])
def test_route_metadata_edges(esmoe, pairs, experts, first, span):
    """Edges of the chunks: a pair per thread, counts taken from the ids up to 8192 pairs and from a launch in front
    past that, more than one round of 1024 pairs per chunk past 262144; skewed ids, some of them -1."""
    from expert_specialization_moe_amd import _native

    rng = np.random.default_rng(pairs)
    ids = (first + np.minimum(rng.geometric(min(0.9, 4.0 / span), size=pairs) - 1, span - 1)).astype(np.int32)
    ids[rng.random(pairs) < 0.05] = -1
    got = _capi_route(_native, ids, first, experts, 256, 128)
    local = (ids >= first) & (ids < first + experts)
    counts = np.bincount(ids[local] - first, minlength=experts)
    offsets, padded = np.concatenate([[0], np.cumsum(counts)]), np.concatenate([[0], np.cumsum((counts + 127) // 128 * 128)])
    dst = np.full(pairs, -1, np.int64)
    order = np.argsort(ids[local], kind="stable")   # local pairs by expert, then by pair index
    dst[np.flatnonzero(local)[order]] = np.arange(order.size)
    assert np.array_equal(got[0], np.stack([counts, np.full(experts, 256), np.full(experts, 128)], axis=1))
    assert np.array_equal(got[1], offsets) and np.array_equal(got[2], padded) and np.array_equal(got[3], dst)


@pytest.mark.parametrize("pairs,experts", [(1000, 32), (1025, 200), (8192, 128), (8193, 128), (300000, 64)])
def test_route_metadata_over_the_ids(esmoe, pairs, experts):
    """Rows written over the ids (one buffer for topk_ids and dst_row): one workgroup, several, several rounds per chunk."""
    from expert_specialization_moe_amd import _native

    ids = np.random.default_rng(pairs).integers(0, experts + 5, size=pairs).astype(np.int32)
    got = _capi_route(_native, ids.copy(), 0, experts, 256, 128, in_place=True)
    ref = oroute.route_metadata(ids, 0, experts, 256, 128)
    for name, g, r in zip(("problem_sizes", "expert_offsets", "blockscale_offsets", "dst_row"), got, ref):
        assert np.array_equal(g, r), name


def test_route_rejects(esmoe):
    from expert_specialization_moe_amd import _native

    p = ctypes.c_void_p(256)
    lib = _native.lib
    assert lib.esmoe_route_metadata(p, 10, 0, 0, 1, 1, p, p, p, p, p, 1 << 20, None) == -1
    assert lib.esmoe_route_metadata(p, 10, 0, 4, 1, 1, p, p, p, p, p, 4, None) == -2
    assert lib.esmoe_permute_rows(p, p, 4, 1, 24, p, None) == -1


@pytest.mark.parametrize("topk,row_elems", [(8, 4096 + 8), (2, 7168), (64, 128), (65, 64), (1, 4104)])
def test_permute_rows_of_topk_pairs(esmoe, topk, row_elems):
    """Row packing for top-k routing (a token's row goes to each of its local pairs' rows, remote pairs skipped),
    rows longer than one 4 KB pass and not a multiple of it; bit-exact against the oracle."""
    tokens, experts = 77, 96
    rng = np.random.default_rng(topk)
    ids = np.stack([rng.permutation(128)[:topk] for _ in range(tokens)]).astype(np.int32)   # experts 96..127 are remote
    x = torch.randn((tokens, row_elems), generator=torch.Generator().manual_seed(topk)).to(torch.bfloat16)
    ps, eo, bso, dst = esmoe.es_route_metadata(torch.from_numpy(ids).cuda(), 0, experts, 256, 128)
    total = int(eo[-1].item())
    packed = torch.full((total, row_elems), float("nan"), dtype=torch.bfloat16, device="cuda")
    esmoe.es_permute_rows(x.cuda(), dst, topk, packed)
    torch.cuda.synchronize()
    ps_r, eo_r, bso_r, dst_r = oroute.route_metadata(ids, 0, experts, 256, 128)
    assert np.array_equal(dst.cpu().numpy(), dst_r)
    assert np.array_equal(H.hp_to_f32(packed.cpu()), oroute.permute_rows(H.hp_to_f32(x), dst_r, topk, total))


@pytest.mark.parametrize("tokens,topk,row_elems", [
    (1, 2, 8), (3, 5, 2048 - 8), (5, 3, 2048), (6, 2, 2048 + 8), (7, 4, 4096), (9, 2, 3 * 2048 + 520),   # around 4096 bytes
    (2100, 2, 4104),             # the same with 3 x 2100 pieces, 52 MB moved
    (4 * (1 << 20) + 5, 2, 8),   # more pieces than one launch takes
])
def test_permute_rows_pieces(esmoe, tokens, topk, row_elems):
    """Rows of one piece, a part of one and several, and a call of more than one launch: a copy, so
    every byte is the source's; rows without a local pair in between, output rows that no pair names untouched."""
    gen = torch.Generator(device="cuda").manual_seed(row_elems + topk)
    x = torch.randint(-30000, 30000, (tokens, row_elems), generator=gen, device="cuda", dtype=torch.int16)
    pairs = tokens * topk
    dst = torch.randperm(pairs, generator=gen, device="cuda").to(torch.int32)
    dst[torch.rand(pairs, generator=gen, device="cuda") < 0.3] = -1
    dst.view(tokens, topk)[tokens // 2] = -1
    out = torch.full((pairs, row_elems), 31000, dtype=torch.int16, device="cuda")
    want = out.clone()
    local = dst >= 0
    want[dst[local].long()] = x[torch.nonzero(local).flatten() // topk]
    esmoe.es_permute_rows(x.view(torch.bfloat16), dst, topk, out.view(torch.bfloat16))
    assert torch.equal(out, want)


@pytest.mark.parametrize("tokens,topk,row_elems,share", [
    (16, 8, 262152, 1.0),        # as many pairs as are looked at, 67 MB packed
    (15, 8, 262152, 1.0),        # fewer
    (4200, 2, 4104, 1.0), (4200, 8, 4104, 0.06), (4200, 8, 4104, 0.5), (4200, 8, 4104, 0.0),
    (2100, 64, 520, 1.0),
])
def test_permute_rows_plain_and_hinted_stores(esmoe, tokens, topk, row_elems, share):
    """Both kinds of stores, chosen by a look at dst_row: the same copy either way."""
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randint(-30000, 30000, (tokens, row_elems), generator=gen, device="cuda", dtype=torch.int16)
    pairs = tokens * topk
    local = torch.rand(pairs, generator=gen, device="cuda") < share
    rows = int(local.sum())
    dst = torch.full((pairs,), -1, dtype=torch.int32, device="cuda")
    dst[local] = torch.randperm(rows, generator=gen, device="cuda").to(torch.int32)
    out = torch.full((rows + 2, row_elems), 31000, dtype=torch.int16, device="cuda")
    want = out.clone()
    want[dst[local].long()] = x[torch.nonzero(local).flatten() // topk]
    esmoe.es_permute_rows(x.view(torch.bfloat16), dst, topk, out.view(torch.bfloat16))
    assert torch.equal(out, want)


def test_routed_fp8_layer_on_device(esmoe):
    """ids -> metadata -> packed rows -> 1x128 quant -> grouped GEMM, all on the device, against the oracle chain."""
    from expert_specialization_moe_amd import workloads as W

    tokens, topk, experts, n, k = 300, 4, 8, 256, 512
    rng = np.random.default_rng(17)
    ids = np.stack([rng.permutation(12)[:topk] for _ in range(tokens)]).astype(np.int32)   # experts 8..11 are remote
    gen = torch.Generator().manual_seed(17)
    x = torch.randn((tokens, k), generator=gen).to(torch.bfloat16)
    w = (torch.randn((experts, n, k), generator=gen) * 0.05).to(torch.bfloat16)
    d_ids = torch.from_numpy(ids).cuda()
    ps, eo, bso, dst = esmoe.es_route_metadata(d_ids, 0, experts, n, k)
    total = int(eo[-1].item())
    packed = torch.full((total, k), float("nan"), dtype=torch.bfloat16, device="cuda")
    esmoe.es_permute_rows(x.cuda(), dst, topk, packed)
    qa, sa = esmoe.es_fp8_quant_act_1x128(packed)
    qw, sw = esmoe.es_fp8_quant_weight_128x128(w.cuda())
    out = torch.full((total, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    stride = torch.full((experts,), k, dtype=torch.int64, device="cuda")
    stride_d = torch.full((experts,), n, dtype=torch.int64, device="cuda")
    esmoe.es_fp8_blockwise_scaled_grouped_mm(out, qa, qw.transpose(1, 2), sa, sw.transpose(1, 2), stride, stride, stride_d,
                                             ps, eo[:experts].contiguous(), torch.empty((0,), dtype=torch.uint8, device="cuda"))
    torch.cuda.synchronize()
    # oracle chain on the host
    ps_r, eo_r, bso_r, dst_r = oroute.route_metadata(ids, 0, experts, n, k)
    assert np.array_equal(ps.cpu().numpy(), ps_r) and np.array_equal(dst.cpu().numpy(), dst_r)
    assert np.array_equal(bso.cpu().numpy(), bso_r)
    packed_r = oroute.permute_rows(H.hp_to_f32(x), dst_r, topk, total)
    assert np.array_equal(H.hp_to_f32(packed.cpu()), packed_r)
    qa_r, sa_r = ofp8.quant_act_1x128(packed_r, scale_via_reciprocal=True)
    assert np.array_equal(qa.view(torch.uint8).cpu().numpy(), qa_r)
    qw_r = np.stack([ofp8.quant_weight_128x128(H.hp_to_f32(w[e]), scale_via_reciprocal=True)[0] for e in range(experts)])
    sw_r = np.stack([ofp8.quant_weight_128x128(H.hp_to_f32(w[e]), scale_via_reciprocal=True)[1] for e in range(experts)])
    ref = ofp8.grouped_mm(qa_r, qw_r, sa_r, sw_r, ps_r, eo_r[:experts])
    rows = [int(v) for v in ps_r[:, 0]]
    H.check_grouped(H.f32(out), ref, rows, [int(v) for v in eo_r[:experts]], "routed layer")
