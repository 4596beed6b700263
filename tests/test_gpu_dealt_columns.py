"""The decode product with the rows of W dealt out evenly over the compute units: at the sizes where the share changes, and
at rows that fill no whole share."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(x, w, dtype, want):
    """A float32 sum of Kd products and the wavefronts' partial sums, in float32 each product once rounded too."""
    b = (x.shape[1] + 16) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    return 2 * b if dtype == torch.float32 else b + 2.0 ** -8 * want.abs()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 8, 16])
@pytest.mark.parametrize("N,Kd", [(4096, 2048), (4097, 2048), (5113, 2064), (5120, 3072), (5121, 2048), (6144, 2048), (6150, 2112),
                                  (7167, 2048), (7169, 2048), (5120, 2032)])
def test_dealt_columns(dtype, M, N, Kd):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(N + M)
    x, w = torch.randn(M, Kd, generator=g).cuda().to(dtype), torch.randn(N, Kd, generator=g).cuda().to(dtype)
    out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
    K.skinny_gemm(x, K.Weight(w), out[:M])
    want = x.double() @ w.double().t()
    assert bool((out[M] == 7.0).all())
    assert bool(((out[:M].double() - want).abs() <= _bound(x, w, dtype, want)).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 9, 16])
@pytest.mark.parametrize("H,KVH,hd,Kd", [(12, 2, 32, 256), (32, 16, 64, 2048), (33, 16, 64, 64), (24, 8, 128, 3072), (25, 8, 128, 512),
                                         (32, 8, 128, 2048), (33, 8, 128, 96), (20, 4, 160, 2560)])
def test_dealt_pairs_turn_and_land_in_their_pages(dtype, M, H, KVH, hd, Kd):
    """Against the product stored and the rotation kernel behind it, whose sums may be taken in another order."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(H * hd + M)
    N, PS = (H + 2 * KVH) * hd, 8
    x, w = torch.randn(M, Kd, generator=g).cuda().to(dtype), torch.randn(N, Kd, generator=g).cuda().to(dtype)
    angle = torch.randn(64, hd // 2, generator=g).cuda()
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, 64, (M,), generator=g).int().cuda()
    slots = torch.randperm(4 * PS, generator=g)[:M].int().cuda()
    slots[M // 2] = -1 if M > 1 else slots[0]            # a row that leaves nothing in the cache
    kp, vp = (torch.full((4, KVH, PS, hd), 3.0, device="cuda", dtype=dtype) for _ in range(2))
    q = K.skinny_qkv_rope(x, K.Weight(w), pos, cos, sin, slots, kp, vp, H, KVH, hd)
    z = (x.double() @ w.double().t()).view(M, H + 2 * KVH, hd)
    b = _bound(x, w, torch.float32, z).view(M, H + 2 * KVH, hd)      # of the sums, before rounding to the type
    c, s = cos.double()[pos.long()][:, None], sin.double()[pos.long()][:, None]
    half, turned = hd // 2, H + KVH
    lo, hi, blo, bhi = z[:, :turned, :half], z[:, :turned, half:], b[:, :turned, :half], b[:, :turned, half:]
    want = torch.cat([torch.cat([lo * c - hi * s, lo * s + hi * c], dim=2), z[:, turned:]], dim=1)
    # the sums' own error turned, and three float32 roundings of the turn's terms, or the rounding to bfloat16
    eps = 2.0 ** -22 if dtype == torch.float32 else 2.0 ** -8
    turn = lambda p, r: torch.cat([p * c.abs() + r * s.abs(), p * s.abs() + r * c.abs()], dim=2)
    tol = torch.cat([turn(blo + eps * lo.abs(), bhi + eps * hi.abs()), b[:, turned:] + eps * z[:, turned:].abs()], dim=1)
    assert bool(((q.view(M, H, hd).double() - want[:, :H]).abs() <= tol[:, :H]).all())
    kept = torch.ones(4 * PS, dtype=torch.bool, device="cuda")
    for m in range(M):
        sl = int(slots[m])
        if sl < 0:
            continue
        kept[sl] = False
        for pool, first in ((kp, H), (vp, turned)):
            got = pool[sl // PS, :, sl % PS].double()
            assert bool(((got - want[m, first:first + KVH]).abs() <= tol[m, first:first + KVH]).all())
    for pool in (kp, vp):
        assert bool((pool.permute(0, 2, 1, 3).reshape(4 * PS, -1)[kept] == 3.0).all())
