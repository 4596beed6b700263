"""Which float32 products go to the one in half precision, and which routed experts go one by one: the rules alone, without a GPU."""
import pytest
import torch

from nanoinfer_amd import kernels as K


class Held:
    """A matrix that counts as kept as pairs of halves."""

    def __init__(self, N, Kd):
        self.rows, self.pairs, self.pair_lines = torch.empty(N, Kd), (None, None), K.pair_lines(N, Kd)


def rows(M, Kd, halved):
    x = torch.empty(M, Kd)
    return K.HalvedRows(x, None, None) if halved else x


@pytest.mark.parametrize("N,Kd,plain,halved", [(16384, 2048, 65, 65), (2048, 8192, 128, 65), (2048, 16384, 112, 65), (3072, 2048, 191, 159),
                                               (2048, 2048, 287, 239), (4096, 14336, 65, 65), (3072, 8192, 86, 65)])
def test_from_how_many_rows(N, Kd, plain, halved):
    """Under 128 rows a product whose x needs a pass of its own takes more work to go there."""
    w = Held(N, Kd)
    assert w.pair_lines[:2] == (plain, halved)
    for M in (65, plain - 1, plain, halved - 1, halved, 128, 2000):
        assert K.pair_wins(rows(M, Kd, False), w) == (M >= plain) or M < 65
        assert K.pair_wins(rows(M, Kd, True), w) == K.takes_halved(M, Kd, torch.float32, w) == (M >= halved)
    assert not K.pair_wins(rows(2000, Kd, False).bfloat16(), w) and not K.takes_halved(2000, Kd, torch.bfloat16, w)
    assert not K.pair_wins(rows(64, Kd, True), w) and not K.takes_halved(w.pair_lines[2] + 1, Kd, torch.float32, w)
    assert not K.pair_wins(rows(2000, Kd, False), w.rows)


@pytest.mark.parametrize("pairs", [True, False])
def test_experts_of_few_rows_stay_together(pairs):
    """Expert by expert is some five launches more: from 128 rows on, whichever products make them."""
    up, down = Held(16 * 2048, 2048), Held(2048, 16 * 1024)
    if not pairs:
        up, down = up.rows, down.rows
    wins = [K.experts_grouped_wins(rows(M, 2048, False), up, down, 4, 16) for M in (65, 96, 127, 300, 1500)]
    assert wins == [False, False, False, True, True]


@pytest.mark.parametrize("M,N,Kd,sums", [(700, 2048, 2048, 4), (1300, 2048, 8192, 3), (1999, 5120, 3072, 3), (2048, 5120, 3072, 3), (600, 16384, 3072, 3),
                                         (448, 6144, 4096, 3), (192, 8192, 2048, 4), (1300, 2048, 4096, 3), (1000, 1536, 1536, 3), (512, 2048, 2048, 4)])
def test_of_how_many_partial_sums_a_result_is_made(M, N, Kd, sums):
    """A plan does not make its sums longer, each of their additions rounded, than plans did when a share was one sum: shares that are not empty, and the
    sums that the tile has for each of them."""
    tile, shares = K.pair_plan(M, N, Kd)[:2]
    per = -(-Kd // (32 * shares)) * 32
    assert -(-Kd // per) * (1 if tile == 0 else 2) >= sums
