"""The rules by which a product goes to a kernel here or to the library, without a GPU."""
import pytest
import torch

from nanoinfer_amd import kernels as K


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 20, 64, 65, 100, 512, 1000])
@pytest.mark.parametrize("N,Kd", [(64, 0), (0, 64)])
def test_products_over_nothing_are_the_librarys(dtype, M, N, Kd):
    """No kernel here takes rows of no elements (it would read the last piece of a row that has none) or none of them."""
    x, weight = torch.empty(M, Kd, dtype=dtype), K.Weight(torch.empty(N, Kd, dtype=dtype))
    if Kd == 0:
        assert not K.skinny_ok(M, Kd, dtype) and not K.skinny_wins(M, Kd, dtype, weight) and not K.skinny_deals(M, N, Kd, dtype, weight)
    assert not K.tiled_wins(x, weight) and not K.tiled_wins(x, weight, gated=True) and not K.split_wins(x, weight.rows)


def test_what_the_tiled_product_cannot_address_is_the_librarys():
    """Bytes of x and of W are counted in 32 bits: what tiled_gemm refuses, the rule does not send there."""
    class Stored:                                      # a matrix that is only looked at
        tiles = torch.empty(0)

        def __init__(self, N, Kd):
            self.rows = torch.empty(N, Kd, dtype=torch.bfloat16, device="meta")

    for M, N, Kd in ((1024, 32, 1 << 20), (512, 4, 1 << 21), (65, 1 << 14, 1 << 16)):
        x = torch.empty(M, Kd, dtype=torch.bfloat16, device="meta")
        assert not K.tiled_wins(x, Stored(N, Kd)) and not K.tiled_wins(x, Stored(N, Kd), gated=True)


def test_a_plan_is_made_once_for_64_rows():
    """Steps of every number of rows weigh the tiles and shares of a product eight times up to 512 rows, not 448 times."""
    from nanoinfer_amd.kernels import tile
    for plan, made in ((K.tiled_plan, tile._tiled_plan), (K.split_plan, tile._split_plan), (lambda M, N, Kd: tile._grouped_plan(M, N, Kd, 7), tile._grouped_tiles)):
        before = made.cache_info().misses
        plans = [plan(M, 3075, 2047) for M in range(65, 513)]
        assert made.cache_info().misses - before <= 8
        assert plans[0] == plan(128, 3075, 2047) and plans[-1] == plan(449, 3075, 2047)
