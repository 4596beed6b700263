"""Hidden units of numbers that are not finite: what comes out is what the formula has, an infinity or NaN, and no finite number."""
import pytest
import torch

pytestmark = pytest.mark.gpu

VALUES = (float("nan"), float("inf"), float("-inf"), 3.0, -3.0, 0.0, -0.0, 0.5)


def same(got, want):
    got, want = got.double().cpu(), want.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    fine = torch.isfinite(want)
    assert torch.allclose(got[fine], want[fine], rtol=1e-2, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ff", [8, 5])                # a thread takes eight numbers or one
def test_experts_act(dtype, ff):
    from nanoinfer_amd import kernels as K
    pairs = torch.tensor([(g, u) for g in VALUES for u in VALUES])
    g, u = pairs[:, :1].expand(-1, ff), pairs[:, 1:].expand(-1, ff)
    mix = torch.full((64, 1), 0.5)
    for up, form, want in ((u.contiguous(), "relu2", torch.relu(u.double()) ** 2),
                           (torch.cat([g, u], 1).contiguous(), "capped_glu", None)):
        if want is None:
            gc, uc = g.double().clamp(max=2.0), u.double().clamp(-2.0, 2.0)
            want = gc / (1.0 + torch.exp(-1.5 * gc)) * (uc + 1.0)
        same(K.experts_act(up.to(dtype).cuda(), mix.cuda(), ff, form, 2.0, 1.5), 0.5 * want)


@pytest.mark.parametrize("M", [1, 20, 100])            # the skinny product's kernels
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_squared_relu_behind_a_product(M, dtype):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, 64, generator=g).to(dtype), torch.randn(48, 64, generator=g).to(dtype)
    x[M - 1, 3], w[5, 7] = float("nan"), float("nan")
    same(K.linear_relu2(x.cuda(), K.Weight(w.cuda())), torch.relu(x.double() @ w.double().t()) ** 2)


def test_few_rows_through_the_chosen_experts():
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(2)
    x, chosen = torch.randn(3, 32, generator=g), torch.tensor([[0, 1], [1, 2], [2, 0]], dtype=torch.int32)
    x[1, 4] = float("nan")
    for form, per in (("relu2", 16), ("capped_glu", 32)):
        up, down = torch.randn(3 * per, 32, generator=g), torch.randn(32, 3 * 16, generator=g)
        got = K.experts_few(x.cuda(), up.cuda(), down.cuda(), chosen.cuda(), torch.full((3, 2), 0.5).cuda(), 16, form, limit=2.0, slope=1.5)
        assert torch.isnan(got).all(dim=1).tolist() == [False, True, False] and bool(torch.isfinite(got[[0, 2]]).all())
