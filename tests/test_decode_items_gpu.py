"""The decode kernel that finishes the q/k/v product: more items of queries, key and value than a block has threads (15 and 16 query
heads of 128 elements with the token's own position), and as many parts of the product as are asked for together, one more, and the
most there are. The same bits as the kernels it stands for."""

from __future__ import annotations

import pytest
from test_kernels_gpu import test_attn_decode_finishes_the_qkv_product_itself as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nkv", [(15, 1), (32, 2), (14, 1)])
@pytest.mark.parametrize("ks,bias,alone", [(8, True, True), (9, False, False), (12, True, False)])
def test_items_and_parts(nq, nkv, ks, bias, alone):
    check(nq, nkv, 128, 16, ks, bias, 0, None, alone)


@pytest.mark.parametrize("nq,nkv,hd,page", [(14, 2, 64, 16), (7, 1, 32, 32), (12, 2, 96, 16), (14, 2, 128, 64)])
@pytest.mark.parametrize("window,size", [(0, None), (0, 3), (70, None), (0, 40)])
def test_forms_that_share_a_unit(nq, nkv, hd, page, window, size):
    """Waves of no, one, two and many chunks, with one set of registers (heads of more than 64 elements) and with two."""
    check(nq, nkv, hd, page, 2, True, window, size, False)


@pytest.mark.parametrize("ks", [1, 4, 5, 8, 12])
@pytest.mark.parametrize("alone", [True, False])
def test_parts_of_small_heads(ks, alone):
    """Heads of 32 elements ask for four parts together where five blocks share a unit."""
    check(7, 1, 32, 16, ks, True, 0, None, alone)
