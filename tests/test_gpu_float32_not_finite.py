"""Float32 prompt attention over keys and queries that are not finite, or too large for a bfloat16, wherever they lie: at the
diagonal, at a window's edge, in prompts shorter than a step of keys, with and without runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

INF, NAN, LARGE = float("inf"), float("nan"), 3.4e38


def attention(q, k, v, scale, window, nsplit):
    """q [T, H, hd] behind the last of k and v [keys, KVH, hd], through pages of 16."""
    from nanoinfer_amd import kernels as K
    (T, H, hd), (keys, KVH) = q.shape, k.shape[:2]
    pages = (keys + 15) // 16
    pools = []
    for t in (k, v):
        padded = torch.zeros(pages * 16, KVH, hd)
        padded[:keys] = t
        pools.append(padded.view(pages, 16, KVH, hd).permute(0, 2, 1, 3).contiguous().cuda())
    qkv = torch.zeros(T, (H + 2 * KVH) * hd)
    qkv[:, :H * hd] = q.reshape(T, H * hd)
    tile = K.mfma_tile_tokens(hd, H // KVH, dtype=torch.float32)
    tiles = torch.tensor(K.build_q_tiles([0], [T], [keys], tile), dtype=torch.int32).view(-1, 4).cuda()
    out = torch.full((T, H * hd), 7.0, device="cuda")            # (a row that is left as it was would show)
    ws = torch.empty(T * H * nsplit * (hd + 2), device="cuda")
    table = torch.arange(pages, dtype=torch.int32).view(1, -1).cuda()
    K.mfma_attention(qkv.cuda(), *pools, table, tiles, out, H, KVH, hd, scale, window, nsplit, ws, tile)
    return out.view(T, H, hd).cpu()


def plain(q, k, v, scale, window):
    """The same in 64 bits over the keys that a row sees.  A score of plus infinity and no score but minus infinity leave a row
    without an answer: NaN."""
    (T, H, hd), (keys, KVH) = q.shape, k.shape[:2]
    out = torch.empty(T, H, hd, dtype=torch.float64)
    for t in range(T):
        n = keys - T + t + 1
        lo = max(0, n - window) if window else 0
        for h in range(H):
            s = (k[lo:n, h // (H // KVH)].double() * q[t, h].double() * scale).sum(-1)
            out[t, h] = torch.softmax(s, 0) @ v[lo:n, h // (H // KVH)].double()
    return out


def check(q, k, v, scale, window, nsplit):
    want = plain(q, k, v, scale, window)
    got = attention(q, k, v, scale, window, nsplit)
    assert torch.equal(got.isnan(), want.isnan())
    # sums of at most some hundred weighted numbers of unit size in 24 bits
    assert float((got.double() - want).nan_to_num().abs().max()) <= 1e-5
    return want


def operands(hd, H, KVH, T, keys):
    g = torch.Generator().manual_seed(31 * T + keys + hd)
    q = torch.randn(T, H, hd, generator=g)
    q[:, :, 9] = torch.where(q[:, :, 9] < 0, -0.02, 0.02)        # (a product with the largest numbers stays finite)
    return q, torch.randn(keys, KVH, hd, generator=g), torch.randn(keys, KVH, hd, generator=g)


SHAPES = [(64, 4, 1), (128, 3, 1), (48, 2, 2), (256, 2, 1)]


@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("value", [INF, -INF, LARGE, -LARGE, NAN])
@pytest.mark.parametrize("hd,H,KVH", SHAPES)
def test_a_spoiled_key(hd, H, KVH, value, nsplit):
    """At the diagonal, a step of keys before it and at a window's edge: rows that see the key have its score, the others none."""
    T, keys, scale = 37, 100, hd ** -0.5
    for at in (keys - 1, keys - 20, keys - T, 65, 40):
        for window in (None, 30):
            q, k, v = operands(hd, H, KVH, T, keys)
            k[at, 0, 9] = value
            want = check(q, k, v, scale, window, nsplit)
            assert at != keys - 1 or not want[:-1].isnan().any()


@pytest.mark.parametrize("nsplit", [1, 2])
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31])
@pytest.mark.parametrize("hd,H,KVH", SHAPES)
def test_prompts_shorter_than_a_step(hd, H, KVH, T, nsplit):
    """Every key lies at the edge of its rows' range."""
    for value in (INF, -INF, LARGE, NAN):
        for at in {0, T // 2, T - 1}:
            q, k, v = operands(hd, H, KVH, T, T)
            k[at, :, 9] = value
            check(q, k, v, hd ** -0.5, None, nsplit)


@pytest.mark.parametrize("nsplit", [1, 3])
@pytest.mark.parametrize("T,keys", [(1, 1), (5, 5), (31, 31), (33, 120)])
@pytest.mark.parametrize("hd,H,KVH", SHAPES)
def test_a_spoiled_query(hd, H, KVH, T, keys, nsplit):
    """Its row has no answer, the others have theirs."""
    for value in (INF, -INF, NAN):
        q, k, v = operands(hd, H, KVH, T, keys)
        q[T // 2, 0, 3] = value
        k[:, :, 3] = torch.where(k[:, :, 3] < 0, -1.0, 1.0)
        k[0, :, 3] = 1.0 if value == INF else -1.0               # at least one score of plus infinity
        want = check(q, k, v, hd ** -0.5, None, nsplit)
        assert want[T // 2, 0].isnan().all() and int(want.isnan().sum()) == hd


@pytest.mark.parametrize("nsplit", [1, 2])
@pytest.mark.parametrize("T,keys", [(9, 9), (20, 75)])
def test_scores_far_below_any_reference(T, keys, nsplit):
    """Every score of a row at -1e32 and less: the one that is largest has all the weight."""
    hd, H, KVH = 64, 2, 1
    q, k, v = operands(hd, H, KVH, T, keys)
    q[:, :, 9] = 1.0
    k[:, :, 9] = -1e33 * (1.0 + torch.arange(keys)[:, None])
    check(q, k, v, hd ** -0.5, None, nsplit)
