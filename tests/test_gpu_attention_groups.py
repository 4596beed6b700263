"""Bfloat16 prompt attention by two groups of wavefronts a tile, each with one half of its keys, against 64 bits of the same rounded
numbers: key ranges of one step (a group without keys), of many segments, cut into runs, windows, several portions."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(portions, H, KVH, hd, ps, blocks, nsplit, window, seed):
    """``portions``: (tokens, keys) of every sequence.  The largest excess over the bound of rounded weights."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(seed)
    T = sum(n for n, _ in portions)
    q = torch.randn(T, H, hd, generator=g).bfloat16()
    counts = [(keys + ps - 1) // ps for _, keys in portions]
    order = torch.randperm(sum(counts) + 1, generator=g)
    kp, vp = (torch.full((len(order), KVH, ps, hd), float("nan"), dtype=torch.bfloat16) for _ in range(2))
    table = torch.zeros(len(portions), max(counts), dtype=torch.int32)
    keys_of, at = [], 0
    for s, (n, keys) in enumerate(portions):
        k, v = (torch.randn(keys, KVH, hd, generator=g).bfloat16() for _ in range(2))
        keys_of.append((k, v))
        mine = order[at:at + counts[s]]
        at += counts[s]
        table[s, :counts[s]] = mine.int()
        for pool, t in ((kp, k), (vp, v)):
            padded = torch.full((counts[s] * ps, KVH, hd), 1.0, dtype=torch.bfloat16)       # a page's unused places hold numbers
            padded[:keys] = t
            pool[mine] = padded.view(counts[s], ps, KVH, hd).permute(0, 2, 1, 3)
    starts = [sum(n for n, _ in portions[:s]) for s in range(len(portions))]
    tile = K.mfma_tile_tokens(hd, H // KVH) * blocks
    tiles = torch.tensor(K.build_q_tiles(starts, [n for n, _ in portions], [c for _, c in portions], tile), dtype=torch.int32).view(-1, 4).cuda()
    qkv = torch.zeros(T, (H + 2 * KVH) * hd, dtype=torch.bfloat16)
    qkv[:, :H * hd] = q.reshape(T, H * hd)
    out = torch.full((T + 1, H * hd), 7.0, device="cuda", dtype=torch.bfloat16)
    ws = torch.empty(T * H * nsplit * (hd + 2), device="cuda")
    K.mfma_attention(qkv.cuda(), kp.cuda(), vp.cuda(), table.cuda(), tiles, out[:T], H, KVH, hd, hd ** -0.5, window, nsplit, ws, tile, 2)
    assert bool((out[T] == 7.0).all())
    got = out[:T].view(T, H, hd).cpu().double()
    worst = -1.0
    for s, (n, keys) in enumerate(portions):
        k, v = keys_of[s]
        for t in sorted({0, 1, n // 2, n - 1}):
            p = keys - n + t
            lo = 0 if window is None else max(0, p + 1 - window)
            for h in range(H):
                kv = h // (H // KVH)
                w = torch.softmax((k[lo:p + 1, kv].double() @ q[starts[s] + t, h].double()) * hd ** -0.5, 0)
                want = w @ v[lo:p + 1, kv].double()
                # weights rounded to 8 bits, in the sum as well; the result's rounding; a score's 2^-24 a product
                bound = 2.0 ** -8 * float(v.abs().max()) + 2.0 ** -8 * want.abs() + 1e-3
                worst = max(worst, float(((got[starts[s] + t, h] - want).abs() - bound).max()))
    return worst


@pytest.mark.parametrize("hd,H,KVH,blocks", [(64, 8, 2, 1), (64, 8, 2, 2), (16, 3, 1, 2), (48, 5, 1, 1), (96, 4, 2, 1), (128, 3, 1, 1)])
@pytest.mark.parametrize("portions,ps,nsplit,window", [
    (((20, 20),), 16, 1, None),                     # tiles of one step: the second group has none
    (((70, 70),), 16, 1, None), (((33, 97),), 16, 1, None), (((65, 200), (3, 40), (17, 17)), 12, 1, None),
    (((40, 2000),), 1, 1, None),                    # three segments of the page table
    (((40, 700),), 16, 3, None), (((20, 65),), 16, 2, None), (((90, 300),), 32, 1, 50)])
def test_two_groups(hd, H, KVH, blocks, portions, ps, nsplit, window):
    assert run(portions, H, KVH, hd, ps, blocks, nsplit, window, hd + blocks) <= 0.0


def test_one_workgroup_for_a_long_and_a_short_tile():
    assert run(((1530, 1530),), 32, 8, 64, 16, 2, 1, None, 5) <= 0.0


@pytest.mark.parametrize("hd,H,KVH,blocks", [(64, 32, 8, 1), (64, 32, 8, 2), (128, 24, 8, 1)])
def test_runs_without_keys_behind_runs_with_keys(hd, H, KVH, blocks):
    """More tiles than the chip holds workgroups, cut into more runs than the short ones have steps: a workgroup goes from a long
    tile to one that is empty for it while its first group may still be taking over the long one's sums."""
    portions = tuple((80, 80 + 640 * (s % 2)) for s in range(16))
    assert run(portions, H, KVH, hd, 16, blocks, 8, None, 11) <= 0.0


def test_the_rule():
    from nanoinfer_amd import kernels as K
    plan = K.mfma_group_plan
    assert plan(64, 4, 8, 512, 512, 512) == (16, 1) == plan(64, 4, 8, 512, 512, 1024)
    assert plan(64, 4, 8, 512, 512, 1100) is None and plan(64, 4, 8, 256, 256, 256) is None
    assert plan(64, 4, 8, 256, 256, 2048) == (16, 2) and plan(64, 4, 8, 1024, 1024, 1024) is None
    assert plan(64, 4, 8, 1024, 1024, 2048) == (32, 1) == plan(64, 4, 8, 1999, 1999, 1999) == plan(64, 4, 8, 3000, 3000, 3000)
    assert plan(64, 4, 8, 1024, 1024, 4096) == (32, 1) and plan(64, 4, 8, 1024, 1024, 4097) is None
    assert plan(64, 4, 8, 4096, 4096, 4096) is None and plan(64, 4, 8, 2048, 2048, 6000) is None
    assert plan(64, 4, 8, 512, 481, 1100) is None                    # several portions in the step
    assert plan(128, 3, 8, 512, 512, 512) is None and plan(128, 3, 8, 512, 512, 2048) == (16, 1)
    with pytest.raises(K.KernelError):
        K.mfma_attention(torch.zeros(1, 768, device="cuda"), *[None] * 5, 1, 1, 256, 1.0, None, groups=2)
