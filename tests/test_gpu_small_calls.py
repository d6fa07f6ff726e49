"""The kernels around the GEMMs where a call is small: the edges of their small forms, against the same oracles as the large ones."""
import pytest
import torch

from tests import test_gpu_fp8_quant_act as A
from tests import test_gpu_routing as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pairs,experts,first,span", [(1, 1024, 0, 1024), (64, 65, 0, 65), (65, 64, 2, 70), (961, 7, 0, 9), (1024, 1024, 3, 1500),
                                                      (1025, 40, 0, 40)])
def test_route_metadata_of_one_workgroup(esmoe, pairs, experts, first, span):
    """Up to 1024 pairs: as many wavefronts as hold the pairs or the experts, the counts from the wavefronts' own pairs."""
    R.test_route_metadata_edges(esmoe, pairs, experts, first, span)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 4096), (3, 640), (1024, 4096), (1025, 4096)])
def test_quant_act_of_resident_launches(esmoe, dtype, shape):
    """One 16-byte load per lane up to 1024 x 4096 values, four past that."""
    A.test_quant_act_bit_exact(esmoe, dtype, shape)


@pytest.mark.parametrize("tokens,topk,row_elems", [(1, 2, 504), (3, 64, 520), (512, 2, 2040), (513, 2, 2040), (256, 2, 2056), (257, 3, 2056), (130, 2, 3 * 2048 + 520)])
def test_permute_rows_on_both_sides_of_the_small_form(esmoe, tokens, topk, row_elems):
    """Pieces of 1024 bytes up to 512 of 4096, of 4096 past that: rows that end inside a piece and inside a load."""
    R.test_permute_rows_pieces(esmoe, tokens, topk, row_elems)
