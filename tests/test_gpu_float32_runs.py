"""Float32 prompt attention with the key ranges cut as the rule cuts them: at the numbers of keys and tiles where it changes,
with runs that some tiles leave empty."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,H,KVH,T,keys,window", [(64, 8, 2, 20, 255, None), (64, 8, 2, 20, 256, None), (64, 8, 2, 33, 300, 40), (64, 8, 2, 33, 300, 250),
                                                    (32, 6, 1, 32, 400, None), (128, 6, 2, 70, 700, None), (64, 32, 8, 260, 260, None),
                                                    (64, 32, 8, 600, 640, 100), (64, 32, 8, 500, 640, 100), (256, 4, 1, 30, 500, None), (48, 5, 5, 17, 1000, 300)])
def test_runs_of_the_rule(hd, H, KVH, T, keys, window):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(T + keys)
    PS, pages = 16, (keys + 15) // 16
    q = torch.randn(T, (H + 2 * KVH) * hd, generator=g).cuda()
    kp, vp = (torch.randn(pages, KVH, PS, hd, generator=g).cuda() for _ in range(2))
    order = torch.randperm(pages, generator=g)
    table = order.int().view(1, -1).cuda()
    tile = K.mfma_tile_tokens(hd, H // KVH, dtype=torch.float32)
    tiles = torch.tensor(K.build_q_tiles([0], [T], [keys], tile), dtype=torch.int32).view(-1, 4).cuda()
    counted = keys if window is None else min(keys, window + T)
    runs = K.mfma_splits(tiles.shape[0], KVH, H // KVH, counted, hd, torch.float32)
    assert (runs > 1) == (counted >= 256)
    out = torch.full((T + 1, H * hd), 7.0, device="cuda")
    ws = torch.full((T * H * runs * (hd + 2),), float("nan"), device="cuda")      # what a run leaves behind it has written itself
    K.mfma_attention(q, kp, vp, table, tiles, out[:T], H, KVH, hd, hd ** -0.5, window, runs, ws, tile)
    k, v = (p[order.cuda()].permute(1, 0, 2, 3).reshape(KVH, pages * PS, hd)[:, :keys].double() for p in (kp, vp))
    at = torch.arange(keys - T, keys, device="cuda")[:, None]
    key = torch.arange(keys, device="cuda")[None]
    seen = (key <= at) & (key > at - (window or keys + 1))
    qh = q[:, :H * hd].double().view(T, KVH, H // KVH, hd)
    s = torch.matmul(qh.permute(1, 2, 0, 3), k.transpose(1, 2).contiguous()[:, None]) * hd ** -0.5
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), dim=-1)
    want = torch.matmul(p, v[:, None]).permute(2, 0, 1, 3).reshape(T, H * hd)
    # a score's error moves a weight by as much of itself: hd + 4 roundings of the score's terms; and one per key of the sums
    size = (qh.abs().permute(1, 2, 0, 3) @ k.abs().transpose(1, 2).contiguous()[:, None]).amax().item() * hd ** -0.5
    bound = 2.0 ** -24 * (2 * (hd + 4) * size + keys + 64) * v.abs().max().item()
    assert float((out[:T].double() - want).abs().max()) <= bound
    assert bool((out[T] == 7.0).all())
