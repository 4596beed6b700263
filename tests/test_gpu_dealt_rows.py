"""The skinny product with more rows than a workgroup holds: rows dealt out to several, at the edges of rows, tiles and pieces."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,Kd", [(65, 16, 16), (96, 17, 48), (97, 100, 192), (129, 256, 512), (256, 1000, 192), (700, 3, 96), (449, 1024, 160), (2049, 33, 64)])
def test_dealt_rows_are_the_rows_alone(dtype, M, N, Kd):
    """Every row gets bit for bit what it gets in a product of the 32 or 64 rows around it that a workgroup takes, whatever
    else is dealt out (a rest of up to 16 rows alone goes to another kernel)."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, Kd, generator=g).cuda().to(dtype), K.Weight(torch.randn(N, Kd, generator=g).cuda().to(dtype))
    types = (torch.float32, dtype) if dtype != torch.float32 else (dtype,)
    for out_type in types:
        out = torch.full((M + 1, N), 7.0, device="cuda", dtype=out_type)
        K.skinny_gemm(x, w, out[:M])
        assert bool((out[M] == 7.0).all())
        want = x.double() @ w.rows.double().t()
        bound = (Kd + 8) * 2.0 ** -24 * (x.double().abs() @ w.rows.double().abs().t())      # a float32 sum of K exact or once rounded products
        if dtype == torch.float32:
            bound = 2 * bound
        if out_type == torch.bfloat16:
            bound = bound + 2.0 ** -8 * want.abs()
        assert bool(((out[:M].double() - want).abs() <= bound).all())
        block = 32 if (N + 15) // 16 * ((M + 31) // 32) <= 256 else 64
        for a in range(0, M - 16, block):
            part = x[a:a + block].contiguous()
            alone = K.skinny_gemm(part, w, torch.empty(part.shape[0], N, device="cuda", dtype=out_type))
            assert torch.equal(out[a:min(a + block, M)], alone)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,inter", [(65, 16), (130, 48), (250, 512)])
def test_dealt_rows_gated_and_squared(dtype, M, inter):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(inter)
    x, w = torch.randn(M, 96, generator=g).cuda().to(dtype), K.Weight(torch.randn(2 * inter, 96, generator=g).cuda().to(dtype))
    calls = K.library_calls()
    gated, squared = K.linear_swiglu(x, w), K.linear_relu2(x, w)
    assert K.library_calls() == calls
    for a in range(0, M, 64):         # the same kernel on 64 rows and fewer
        b = min(a + 64, M)
        part = x[a:b].contiguous()
        if b - a > 32:
            one = K.skinny_gemm(part, w, torch.empty(b - a, inter, device="cuda", dtype=dtype), swiglu=True)
            assert torch.allclose(gated[a:b].float(), one.float(), rtol=2.0 ** -7 if dtype == torch.bfloat16 else 1e-5, atol=1e-4)
    z = x.double() @ w.rows.double().t()
    want = torch.relu(z) ** 2
    assert float((squared.double() - want).abs().max()) <= (2.0 ** -7 if dtype == torch.bfloat16 else 1e-5) * float(want.abs().max())


def test_what_is_not_dealt():
    from nanoinfer_amd import kernels as K
    x, w = torch.randn(100, 64).cuda(), K.Weight(torch.randn(48, 64).cuda())
    h = torch.zeros(100, 48).cuda()
    for bad in (lambda: K.skinny_gemm(x, w.rows, torch.empty(100, 48).cuda()), lambda: K.skinny_gemm(x, w, h, residual=True),
                lambda: K.skinny_gemm(x, w, torch.empty(100, 24).cuda(), swiglu=True),
                lambda: K.skinny_gemm(x[:, :60].contiguous(), K.Weight(w.rows[:, :60].contiguous()), torch.empty(100, 48).cuda())):
        with pytest.raises(K.KernelError):
            bad()
