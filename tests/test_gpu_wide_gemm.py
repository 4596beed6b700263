"""The bfloat16 products of many rows on both operands as stored (``csrc/wide_gemm.hip``) alone: every tile at its edges, every ring of
stages from its first turn on, every epilogue."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nanoinfer_amd import kernels
    return kernels


def operands(M, N, Kd, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(M, Kd, generator=g).bfloat16().cuda(), torch.randn(N, Kd, generator=g).bfloat16().cuda()


def bound(x, w, rounded):
    """K roundings of at most 2^-24 of sum |x||w|, and one of the result to bfloat16."""
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    return want, (x.shape[1] + 8) * 2.0 ** -24 * size + (2.0 ** -8 * want.abs() if rounded else 0.0)


# rows: one, the edges of 128 and 256, more than a group of four tiles, several of them (each begins at another stage); columns: the
# smallest, edges of 128 and 256; stages of 64: one, fewer than any ring holds, turns and remainders of rings of 2, 3, 5 and 6
@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("M,N,Kd", [(1, 16, 64), (127, 128, 128), (129, 240, 192), (255, 272, 256), (257, 16, 320), (640, 144, 384), (1030, 256, 448),
                                    (1025, 400, 704), (2300, 48, 832)])
def test_every_tile_at_its_edges(K, tile, M, N, Kd):
    x, w = operands(M, N, Kd, seed=M + N + Kd)
    plain = tile if tile < 4 else 3                             # (the other is for products with SwiGLU alone)
    for dtype in (torch.bfloat16, torch.float32):
        out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
        K.wide_gemm(x, w, dtype, out[:M], tile=plain)
        want, most = bound(x, w, dtype == torch.bfloat16)
        assert bool(((out[:M].double() - want).abs() <= most).all())
        assert bool((out[M] == 7.0).all())                       # nothing behind the last row
    sums = K.wide_gemm(x, w, torch.float32, tile=plain)
    assert torch.equal(K.wide_gemm(x, w, torch.float32, squared=True, tile=plain), torch.relu(sums) ** 2)
    if N % 32 == 0:
        half = N // 2
        size = (x.float().abs() @ w.float().abs().t()).double()
        for act in ("silu", "gelu_tanh"):
            out = torch.full((M + 1, half), 7.0, device="cuda", dtype=torch.bfloat16)
            K.wide_gemm(x, w, out=out[:M], gated=act, tile=tile)
            # of the float32 sums of another tile, by the kernel of its own: |d act| <= 1.2 |d gate|, |act| <= |gate|
            want = K.swiglu(sums, torch.empty(M, half, device="cuda"), act).double()
            off = 2 * (Kd + 8) * 2.0 ** -24 * (1.2 * size[:, :half] * sums[:, half:].abs() + size[:, half:] * sums[:, :half].abs())
            assert bool(((out[:M].double() - want).abs() <= 2.0 ** -8 * want.abs() + off + 1e-30).all())
            assert bool((out[M] == 7.0).all())


def test_rows_that_are_not_finite_stay_so_and_touch_no_other(K):
    x, w = operands(300, 256, 128)
    clean = K.wide_gemm(x, w)
    x[3, 5], x[299, 127] = float("inf"), float("nan")
    got = K.wide_gemm(x, w)
    kept = torch.ones(300, dtype=torch.bool)
    kept[[3, 299]] = False
    assert not bool(torch.isfinite(got[~kept.cuda()]).any()) and torch.equal(got[kept.cuda()], clean[kept.cuda()])


def test_products_of_many_rows_go_there_and_beside_no_library(K):
    calls = K.library_calls()
    for M, N, Kd, gated in ((1999, 2048, 2048, False), (1024, 4096, 2048, True), (512, 16384, 2048, True)):
        x, w = operands(M, N, Kd)
        assert K.wide_wins(x, w, gated)
        weight = K.Weight(w, tiled=False)
        if gated:
            got, sums = K.linear_swiglu(x, weight), K.wide_gemm(x, w, torch.float32)
            want = K.swiglu(sums, torch.empty(M, N // 2, device="cuda"))
            assert bool(((got.float() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -12 * sums.abs().max()).all())
        else:
            want, most = bound(x, w, True)
            assert bool(((K.linear(x, weight).double() - want).abs() <= most).all())
            assert torch.equal(K.linear(x, weight, torch.float32), K.wide_gemm(x, w, torch.float32))
            relu2 = K.linear_relu2(x, weight)
            assert torch.equal(relu2, K.wide_gemm(x, w, squared=True))
    assert K.library_calls() == calls


def test_what_it_does_not_take(K):
    x, w = operands(600, 64, 128)
    for bad in (lambda: K.wide_gemm(x[:, :96].contiguous(), w[:, :96].contiguous()), lambda: K.wide_gemm(x, w[:40]), lambda: K.wide_gemm(x, w[:, :64]),
                lambda: K.wide_gemm(x, w[:48], gated="silu"), lambda: K.wide_gemm(x, w, torch.float32, gated="silu"),
                lambda: K.wide_gemm(x, w, out=torch.empty(600 * 64 + 1, device="cuda", dtype=torch.bfloat16)[1:].view(600, 64)),
                lambda: K.wide_gemm(x.float(), w.float()), lambda: K.wide_gemm(x.t().contiguous().t(), w)):
        with pytest.raises(K.KernelError):
            bad()
