"""The products of bfloat16 activations in the tiles that their sizes choose: 64 x 64 by four waves, 64 x 96, 64 x 128, rows and tokens that end inside a tile, one and several stages of K, segments"""
import pytest

from tests.test_dense_rounded import test_products_of_rounded_activations as products


@pytest.mark.gpu
@pytest.mark.parametrize("rows,K,T,segs,act", [(1999, 64, 450, 1, 0), (2044, 320, 450, 1, 1), (2560, 192, 500, 1, 2), (2000, 64, 1001, 1, 0), (1030, 192, 1900, 1, 1), (2020, 512, 1000, 1, 3), (2100, 128, 900, 3, 0)])
def test_products_by_size(rows, K, T, segs, act):
    products(rows, K, T, segs, act)
