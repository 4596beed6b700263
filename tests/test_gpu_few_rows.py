"""Float32 products of four and of eight rows by 4 x 4 blocks: at the numbers of rows and lengths where the kernel changes,
and that the kernels for a matrix as stored and re-tiled add such rows up in the same order where both have eight wavefronts
(rows of fewer than 2,048 elements)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9])
@pytest.mark.parametrize("N,Kd", [(16, 8), (40, 200), (3, 1024), (33, 1032), (1000, 1056), (2049, 2048), (1040, 3080)])
def test_few_rows(M, N, Kd):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(N * M)
    x, w = torch.randn(M, Kd, generator=g).cuda(), torch.randn(N, Kd, generator=g).cuda()
    want = x.double() @ w.double().t()
    tol = 2 * (Kd + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())     # every product and every sum rounded once
    results = []
    for weight in (w, K.Weight(w)):
        out = torch.full((M + 1, N), 7.0, device="cuda")
        K.skinny_gemm(x, weight, out[:M])
        results.append(out)
        assert bool(((out[:M].double() - want).abs() <= tol).all()) and bool((out[M] == 7.0).all())
        stream = torch.randn(M, N, generator=g).cuda()
        if isinstance(weight, K.Weight):
            h = stream.clone()
            K.skinny_gemm(x, weight, h, residual=True)
            assert bool(((h.double() - stream.double() - want).abs() <= tol + 2.0 ** -23 * h.double().abs()).all())
    if Kd < 2048:
        assert torch.equal(*results)
    if N % 32 == 0:
        gated = K.skinny_gemm(x, K.Weight(w), torch.empty(M, N // 2, device="cuda"), swiglu=True)
        a, b = want[:, :N // 2], want[:, N // 2:]
        ref = torch.nn.functional.silu(a) * b
        assert bool(((gated.double() - ref).abs() <= 1.1 * (tol[:, :N // 2] * b.abs() + tol[:, N // 2:] * a.abs()) + 1e-5 * ref.abs() + 1e-6).all())


@pytest.mark.parametrize("M", [1, 4, 8])
def test_a_row_does_not_see_the_others(M):
    """A row with infinities and a row of NaN leave the other rows bit for bit what they are beside zeros."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, 2048, generator=g).cuda(), K.Weight(torch.randn(96, 2048, generator=g).cuda())
    clean = K.skinny_gemm(x, w, torch.empty(M, 96, device="cuda"))
    for bad in range(M):
        for value in (float("inf"), float("nan")):
            y = x.clone()
            y[bad, 5] = value
            out = K.skinny_gemm(y, w, torch.empty(M, 96, device="cuda"))
            rest = [m for m in range(M) if m != bad]
            assert torch.equal(out[rest], clean[rest]) and not bool(torch.isfinite(out[bad]).any())
