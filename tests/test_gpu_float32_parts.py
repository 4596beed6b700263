"""Float32 prompt attention in three bfloat16 parts: what is not finite, or too large for a bfloat16, comes out as the float32
instructions give it; weights far below the reference; halves of tiles without tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def attention(hd, H, KVH, q, k, v, T, nsplit, scale):
    """q [T, H, hd], k and v [keys, KVH, hd] through pages of 16 in a shuffled order."""
    from nanoinfer_amd import kernels as K
    keys = k.shape[0]
    pages = (keys + 15) // 16
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(keys))
    kp, vp = (torch.zeros(pages, KVH, 16, hd) for _ in range(2))
    for pool, t in ((kp, k), (vp, v)):
        padded = torch.zeros(pages * 16, KVH, hd)
        padded[:keys] = t
        pool[order] = padded.view(pages, 16, KVH, hd).permute(0, 2, 1, 3)
    qkv = torch.zeros(T, (H + 2 * KVH) * hd)
    qkv[:, :H * hd] = q.reshape(T, H * hd)
    tile = K.mfma_tile_tokens(hd, H // KVH, dtype=torch.float32)
    tiles = torch.tensor(K.build_q_tiles([0], [T], [keys], tile), dtype=torch.int32).view(-1, 4).cuda()
    out = torch.full((T + 1, H * hd), 7.0, device="cuda")
    ws = torch.empty(T * H * nsplit * (hd + 2), device="cuda")
    K.mfma_attention(qkv.cuda(), kp.cuda(), vp.cuda(), order.int().view(1, -1).cuda(), tiles, out[:T], H, KVH, hd, scale, None, nsplit, ws, tile)
    assert bool((out[T] == 7.0).all())
    return out[:T].view(T, H, hd).cpu()


def plain(q, k, v, T, scale):
    """The same in 64 bits; a key that a row does not see has no part in it."""
    keys, H, KVH = k.shape[0], q.shape[1], k.shape[1]
    out = torch.empty(T, H, q.shape[2], dtype=torch.float64)
    for t in range(T):
        n = keys - T + t + 1
        for h in range(H):
            g = h // (H // KVH)
            s = (k[:n, g].double() @ q[t, h].double()) * scale
            out[t, h] = torch.softmax(s, 0) @ v[:n, g].double()
    return out


def operands(hd, H, KVH, T, keys, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(T, H, hd, generator=g), torch.randn(keys, KVH, hd, generator=g), torch.randn(keys, KVH, hd, generator=g))


@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("hd,H,KVH,T,keys", [(64, 4, 1, 33, 120), (128, 3, 1, 18, 90), (48, 2, 2, 37, 100), (16, 8, 1, 20, 64), (256, 2, 1, 9, 70)])
def test_values_that_are_not_finite(hd, H, KVH, T, keys, nsplit):
    q, k, v = operands(hd, H, KVH, T, keys, hd)
    scale = hd ** -0.5
    want = plain(q, k, v, T, scale)
    v[2, 0, 5], v[3, 0, 6], v[4, 0, 7] = float("inf"), float("-inf"), float("nan")
    v[5, 0, 8] = 3.4e38                                       # rounds to an infinite bfloat16
    spoiled = plain(q, k, v, T, scale)
    got = attention(hd, H, KVH, q, k, v, T, nsplit, scale)
    group = H // KVH
    assert bool((got[:, :group, 5] == float("inf")).all() and (got[:, :group, 6] == float("-inf")).all() and got[:, :group, 7].isnan().all())
    assert torch.allclose(got[:, :group, 8].double(), spoiled[:, :group, 8], rtol=1e-5)
    others = [c for c in range(hd) if c not in (5, 6, 7, 8)]
    assert float((got[:, :, others].double() - want[:, :, others]).abs().max()) <= 1e-5
    assert float((got[:, group:].double() - want[:, group:]).abs().max() if H > group else 0.0) <= 1e-5


@pytest.mark.parametrize("hd,H,KVH", [(64, 4, 1), (128, 3, 1), (32, 2, 1)])
def test_keys_too_large_for_a_bfloat16(hd, H, KVH):
    """One key's score is so large or so small that it is the only weight or none; minus infinity is none (a row with a score of
    plus infinity has no answer)."""
    T, keys, scale = 21, 75, hd ** -0.5
    q, k, v = operands(hd, H, KVH, T, keys, hd + 1)
    q[:, :, 9] = torch.where(q[:, :, 9] < 0, -0.02, 0.02)
    k[1] = 0.0
    k[1, :, 9] = 3.4e38
    want = plain(q, k, v, T, scale)
    got = attention(hd, H, KVH, q, k, v, T, 1, scale)
    assert float((got.double() - want).abs().max()) <= 1e-5
    k[1, :, 9] = float("inf")
    got = attention(hd, H, KVH, q, k, v, T, 1, scale)
    down = (q[:, :, 9] < 0)[..., None].expand_as(got)
    assert bool(down.any()) and float((got.double() - want)[down].abs().max()) <= 1e-5
    k[1, :, 9] = 0.0
    k[1] = k[1] - 1e30                                         # (every row: far below or far above)
    want = plain(q, k, v, T, scale)
    assert float((attention(hd, H, KVH, q, k, v, T, 2, scale).double() - want).abs().max()) <= 1e-5


@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 32, 33])
def test_halves_of_tiles(T):
    """At head size 64 a tile has tokens for two workgroups: the second may have none."""
    hd, H, KVH, keys = 64, 4, 2, 64
    q, k, v = operands(hd, H, KVH, T, keys, T)
    want = plain(q, k, v, T, 0.125)
    assert float((attention(hd, H, KVH, q, k, v, T, 1, 0.125).double() - want).abs().max()) <= 2e-6


def test_weights_far_below_the_reference_keep_their_places():
    """Scores spread over 180: weights down to nothing, their order and sum as in 64 bits."""
    hd, H, KVH, T, keys = 64, 4, 1, 16, 200
    q, k, v = operands(hd, H, KVH, T, keys, 7)
    q, k = q * 0.0, k * 0.0
    q[:, :, 0] = 1.0
    k[:, 0, 0] = torch.linspace(-90.0, 90.0, keys)[torch.randperm(keys, generator=torch.Generator().manual_seed(3))]
    want = plain(q, k, v, T, 1.0)
    got = attention(hd, H, KVH, q, k, v, T, 1, 1.0).double()
    # a weight e^t is off by (|t| + 4) roundings of itself; over weights that fall by e^0.9 a key, numerator and denominator, that
    # is 2 (1 + 4) of the largest value, and a few for the sums
    assert float((got - want).abs().max()) <= 16 * 2.0 ** -24 * float(v.abs().max())


@pytest.mark.parametrize("hd,nsplit", [(256, 2), (256, 3), (160, 3), (128, 3)])
def test_one_run_of_keys_is_made_again(hd, nsplit):
    """The run with a value too large for a bfloat16 goes to the float32 instructions, the others do not: together they have every
    key once, also where those take fewer keys a step."""
    H, KVH, T, keys = 2, 1, 17, 120
    q, k, v = operands(hd, H, KVH, T, keys, hd)
    v[3, 0, 8] = 3.4e38
    want = plain(q, k, v, T, hd ** -0.5)
    got = attention(hd, H, KVH, q, k, v, T, nsplit, hd ** -0.5)
    assert torch.allclose(got[:, :, 8].double(), want[:, :, 8], rtol=1e-5)
    others = [c for c in range(hd) if c != 8]
    assert float((got[:, :, others].double() - want[:, :, others]).abs().max()) <= 1e-5
