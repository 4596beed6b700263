"""17 to 64 bfloat16 rows on a wide matrix as stored (the head over the vocabulary): the tiles of few rows at their edges, and where the rule sends
products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def worst(x, w, got):
    """Largest excess over K roundings of at most 2^-24 of sum |x||w|."""
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    return float(((got.double() - want).abs() - (x.shape[1] + 8) * 2.0 ** -24 * size).max())


# rows: edges of 16, 32 and 64, more than a tile; columns: the smallest, edges of 128 and 256; stages of 64: fewer than the ring holds, its turns and remainders
@pytest.mark.parametrize("tile", [5, 6])
@pytest.mark.parametrize("M,N,Kd", [(1, 16, 64), (17, 128, 128), (33, 240, 192), (63, 272, 256), (64, 256, 320), (65, 144, 384), (300, 400, 448)])
def test_tiles_of_few_rows(tile, M, N, Kd):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, Kd, generator=g).bfloat16().cuda(), torch.randn(N, Kd, generator=g).bfloat16().cuda()
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
        K.wide_gemm(x, w, dtype, out[:M], tile=tile)
        assert bool((out[M] == 7.0).all())                       # nothing behind the last row
        if dtype == torch.float32:
            assert worst(x, w, out[:M]) <= 0.0
            sums = out[:M].clone()
        else:
            assert torch.equal(out[:M], sums.bfloat16())
    with pytest.raises(K.KernelError):
        K.wide_gemm(x, w[:N // 32 * 32], gated="silu", tile=tile)     # no epilogue but a plain store is compiled for them


@pytest.mark.parametrize("M", [16, 17, 40, 64, 65])
@pytest.mark.parametrize("N,Kd,most", [
    (32000, 2048, 64), (32016, 2112, 0), (128256, 2048, 64), (32000, 4096, 0), (32000, 4160, 0), (31984, 2048, 0),
    (36864, 2048, 0), (49152, 2112, 64), (66560, 2112, 32), (98304, 2112, 64), (49152, 4096, 64), (66560, 4096, 0)])
def test_the_head_of_few_rows(M, N, Kd, most):
    """Whichever way a product goes the sums are float32's, into a tensor of its own or a given one, on replays of a recorded launch too."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = (torch.randn(n, Kd, generator=g, device="cuda").bfloat16() for n in (M, N))
    assert K.wide_few_wins(M, Kd, w) == (16 < M <= most)
    out = torch.full((M + 1, N), 7.0, device="cuda")
    assert K.linear(x, w, out_dtype=torch.float32, out=out[:M]) is not None
    assert worst(x, w[::61], out[:M, ::61]) <= 0.0 and worst(x, w[-100:], out[:M, -100:]) <= 0.0
    assert bool((out[M] == 7.0).all())
    assert torch.equal(K.linear(x, w, out_dtype=torch.float32), out[:M])
    odd = torch.empty(M * Kd + 1, device="cuda", dtype=torch.bfloat16)[1:].view(M, Kd)      # rows off sixteen bytes go to the library
    odd.copy_(x)
    assert worst(x, w[-100:], K.linear(odd, w, out_dtype=torch.float32)[:, -100:]) <= 0.0
