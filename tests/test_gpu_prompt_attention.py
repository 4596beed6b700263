"""The bfloat16 prompt attention of head sizes 64 and 128 against 64 bits of the same rounded numbers: where its stages, sets and pages end,
single tokens beside portions, scores that rise far above a row's first ones (the tile is made again), key ranges past the page numbers in LDS."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def worst_excess(portions, H, KVH, hd, ps, blocks=1, groups=1, nsplit=1, window=None, seed=0, plant=None, off=0):
    """``portions``: (tokens, keys) of every sequence.  The largest excess over the bound of rounded weights.  ``off``: elements by which the pools start
    behind an allocation's first byte."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(seed)
    T = sum(n for n, _ in portions)
    counts = [(keys + ps - 1) // ps for _, keys in portions]
    order = torch.randperm(sum(counts) + 1, generator=g)
    kp, vp = (torch.full((len(order), KVH, ps, hd), float("nan"), dtype=torch.bfloat16) for _ in range(2))      # a page of nobody's is no number
    table = torch.full((len(portions), max(counts)), -1, dtype=torch.int32)
    starts = [sum(n for n, _ in portions[:s]) for s in range(len(portions))]
    q = torch.randn(T, H, hd, generator=g).bfloat16()
    keys_of, at = [], 0
    for s, (n, keys) in enumerate(portions):
        k, v = (torch.randn(keys, KVH, hd, generator=g).bfloat16() for _ in range(2))
        if plant is not None:
            plant(q[starts[s]:starts[s] + n], k, v)
        keys_of.append((k, v))
        mine, at = order[at:at + counts[s]], at + counts[s]
        table[s, :counts[s]] = mine.int()
        for pool, t in ((kp, k), (vp, v)):
            padded = torch.full((counts[s] * ps, KVH, hd), float("nan"), dtype=torch.bfloat16)
            padded[:keys] = t
            pool[mine] = padded.view(counts[s], ps, KVH, hd).permute(0, 2, 1, 3)
    tile = K.mfma_tile_tokens(hd, H // KVH) * blocks
    tiles = torch.tensor(K.build_q_tiles(starts, [n for n, _ in portions], [c for _, c in portions], tile), dtype=torch.int32).view(-1, 4).cuda()
    qkv = torch.zeros(T, (H + 2 * KVH) * hd, dtype=torch.bfloat16)
    qkv[:, :H * hd] = q.reshape(T, H * hd)
    out = torch.full((T + 1, H * hd), 7.0, device="cuda", dtype=torch.bfloat16)
    ws = torch.empty(T * H * nsplit * (hd + 2), device="cuda")
    kp, vp = (torch.cat([p.new_zeros(off), p.view(-1)]).cuda()[off:].view(p.shape) for p in (kp, vp))
    K.mfma_attention(qkv.cuda(), kp, vp, table.cuda(), tiles, out[:T], H, KVH, hd, hd ** -0.5, window, nsplit, ws, tile, groups)
    assert bool((out[T] == 7.0).all())
    got, worst = out[:T].view(T, H, hd).cpu().double(), -1.0
    for s, (n, keys) in enumerate(portions):
        k, v = keys_of[s]
        for t in sorted({0, 1, n // 2, n - 2, n - 1} & set(range(n))):
            p = keys - n + t
            lo = 0 if window is None else max(0, p + 1 - window)
            for h in range(H):
                kv = h // (H // KVH)
                w = torch.softmax((k[lo:p + 1, kv].double() @ q[starts[s] + t, h].double()) * hd ** -0.5, 0)
                want = w @ v[lo:p + 1, kv].double()
                here = got[starts[s] + t, h]
                same = (here == want) | (here.isnan() & want.isnan())        # (infinities, where some are planted)
                # weights rounded to 8 bits, in the sum as well; the result's rounding; a score's 2^-24 a product
                biggest = v[lo:p + 1, kv].double().nan_to_num(0.0, 0.0, 0.0).abs().amax(0)         # (of each dim)
                excess = torch.where(same, torch.full_like(want, -1.0), (here - want).abs() - 2.0 ** -8 * biggest - 2.0 ** -8 * want.abs() - 1e-3)
                assert not bool(excess.isnan().any())
                worst = max(worst, float(excess.max()))
    return worst


@pytest.mark.parametrize("hd,H,KVH,blocks,groups", [(64, 4, 1, 1, 1), (64, 8, 2, 2, 1), (64, 4, 1, 2, 2), (64, 5, 1, 1, 2), (128, 3, 1, 1, 1), (128, 4, 2, 1, 2)])
@pytest.mark.parametrize("portions,ps", [
    (((1, 1),), 16), (((31, 31), (33, 64), (2, 65)), 16), (((63, 63),), 32), (((64, 64), (65, 65)), 64), (((40, 127), (9, 129)), 16),
    (((17, 191), (1, 192), (1, 193), (1, 7)), 16), (((130, 500),), 256), (((20, 20480 + 40),), 16),
    (((31, 31), (33, 64), (2, 65), (1, 9)), 8), (((40, 127), (9, 129), (70, 500)), 8)])
def test_ends_of_stages_and_pages(hd, H, KVH, blocks, groups, portions, ps):
    assert worst_excess(portions, H, KVH, hd, ps, blocks, groups, seed=hd + blocks) <= 0.0


@pytest.mark.parametrize("hd,H,KVH,blocks", [(64, 4, 1, 1), (64, 4, 1, 2), (64, 3, 3, 1), (128, 3, 1, 1)])
@pytest.mark.parametrize("window,nsplit", [(1, 1), (31, 1), (64, 1), (65, 1), (200, 1), (200, 2), (1000, 1)])
def test_windows(hd, H, KVH, blocks, window, nsplit):
    """Windows that start and end at and beside stages and sets, rows whose window starts inside the tile's first ones, and one longer than the keys."""
    assert worst_excess(((130, 500), (33, 33), (64, 128)), H, KVH, hd, 16, blocks, nsplit=nsplit, window=window, seed=window) <= 0.0


@pytest.mark.parametrize("hd,H,KVH,groups", [(64, 4, 1, 1), (64, 4, 1, 2), (128, 3, 1, 1)])
@pytest.mark.parametrize("off", [1, 4])
def test_pools_off_sixteen_bytes(hd, H, KVH, groups, off):
    """Views into a program's own buffers: what goes straight into LDS would start between sixteen bytes, so that another kernel takes them."""
    assert worst_excess(((17, 191), (1, 193), (40, 40)), H, KVH, hd, 16, 1, groups, seed=off, off=off) <= 0.0


def test_more_pages_than_their_numbers_in_lds():
    assert worst_excess(((9, 50000),), 4, 1, 64, 16) <= 0.0


@pytest.mark.parametrize("hd,groups", [(64, 1), (64, 2), (128, 1), (128, 2)])
def test_keys_further_than_two_gigabytes(hd, groups):
    """A sequence whose key rows, one behind the other, would pass 2^31 bytes: the few pages behind that hold the keys that count, the others are the
    same 64 pages over and over."""
    from nanoinfer_amd import kernels as K
    ps, H, n, few = 256, 2, 40, 3
    far = (1 << 31) // (2 * hd) // ps                           # the first page past it
    keys = (far + few) * ps
    g = torch.Generator().manual_seed(hd)
    kp, vp = (torch.randn(64 + few, 1, ps, hd, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(n, H, hd, generator=g).bfloat16()
    q[..., 0], kp[..., 0] = 8.0, 0.0
    kp[64:, :, 5::16, 0] = 24.0 * hd ** 0.5 / 8.0               # e^24 of the others, of which there are e^16
    table = torch.cat([torch.arange(far) % 64, 64 + torch.arange(few)]).int().view(1, -1).cuda()
    qkv = torch.zeros(n, (H + 2) * hd, dtype=torch.bfloat16)
    qkv[:, :H * hd] = q.reshape(n, H * hd)
    tile, nsplit = K.mfma_tile_tokens(hd, H), 16
    tiles = torch.tensor(K.build_q_tiles([0], [n], [keys], tile), dtype=torch.int32).view(-1, 4).cuda()
    out, ws = torch.empty(n, H * hd, device="cuda", dtype=torch.bfloat16), torch.empty(n * H * nsplit * (hd + 2), device="cuda")
    K.mfma_attention(qkv.cuda(), kp.cuda(), vp.cuda(), table, tiles, out, H, 1, hd, hd ** -0.5, None, nsplit, ws, tile, groups)
    k, v = (p[:, 0].reshape(-1, hd).double() for p in (kp, vp))
    for t in (0, n - 1):
        rows = keys - n + t + 1
        times = torch.cat([torch.full((64 * ps,), float(far // 64)) + (torch.arange(64 * ps) < far % 64 * ps), (torch.arange(few * ps) < rows - far * ps).double()])
        for h in range(H):
            w = times * torch.exp((k @ q[t, h].double()) * hd ** -0.5 - 24.0)
            want = w @ v / w.sum()
            here = out[t].view(H, hd)[h].cpu().double()
            assert float(((here - want).abs() - 2.0 ** -8 * float(v.abs().max()) - 2.0 ** -8 * want.abs()).max()) <= 1e-3


@pytest.mark.parametrize("hd,H,KVH", [(64, 8, 2), (64, 20, 1), (128, 6, 2)])
@pytest.mark.parametrize("window,nsplit", [(None, 1), (40, 1), (None, 3)])
def test_single_tokens_beside_a_portion(hd, H, KVH, window, nsplit):
    portions = ((70, 70),) + tuple((1, keys) for keys in (1, 31, 32, 33, 128, 129, 700)) + ((2, 300),)
    assert worst_excess(portions, H, KVH, hd, 16, nsplit=nsplit, window=window, seed=3) <= 0.0


def planted(rise, first, every):
    """Keys from ``first`` on that every query likes by e^rise more than the others.  Checked here, in powers of two above the largest score of the first 32
    keys (a walk's reference): what the weights of the keys up to the first planted one's stage sum to lies in float32's ordinary range, or beyond what
    the kernel lets a tile keep without a look at its scores (2^100)."""
    def plant(q, k, v):
        n, hd = len(k), q.shape[-1]
        q[..., 0] = 8.0
        k[..., 0] = 0.0
        k[first::every, :, 0] = rise * hd ** 0.5 / 8.0
        if n > first:
            base = torch.einsum("thd,khd->thk", q[:, ::q.shape[1] // k.shape[1]].double(), k[:first // 64 * 64 + 64].double()) * hd ** -0.5 / math.log(2.0)
            risen = torch.logsumexp(base * math.log(2.0), -1) / math.log(2.0) - base[..., :32].amax(-1)
            assert float(risen.min()) > 101.0 if rise > 70.0 else float(risen.max()) < 97.0, (float(risen.min()), float(risen.max()))
    return plant


@pytest.mark.parametrize("hd,blocks,groups", [(64, 1, 1), (64, 1, 2), (64, 2, 1), (64, 2, 2), (128, 1, 1), (128, 1, 2)])
@pytest.mark.parametrize("nsplit,rise", [(1, 3.0), (1, 20.0), (2, 20.0), (1, 60.0), (2, 60.0), (1, 80.0), (2, 80.0), (1, 120.0), (2, 120.0)])
def test_scores_that_rise_late(hd, blocks, groups, nsplit, rise):
    """Up to e^60 the weights stay in the range that a tile is kept with; past e^69 it is made again, with e^80 from sums that are numbers, with e^120 from
    infinities."""
    assert worst_excess(((150, 400), (60, 60)), 4, 2, hd, 16, blocks, groups, nsplit, seed=5, plant=planted(rise, 100, 37)) <= 0.0


@pytest.mark.parametrize("hd,blocks", [(64, 1), (64, 2), (128, 1)])
@pytest.mark.parametrize("rise", [20.0, 60.0, 80.0, 120.0])
def test_scores_that_rise_late_in_a_window(hd, blocks, rise):
    """The sets between a window's edges are not looked at either (their first keys here are some of the sequence's)."""
    assert worst_excess(((150, 900), (60, 60)), 4, 2, hd, 16, blocks, window=700, seed=8, plant=planted(rise, 600, 37)) <= 0.0


@pytest.mark.parametrize("groups", [1, 2])
def test_values_that_are_not_finite(groups):
    """An infinity in one dim of one value is in that dim of every row that reads it and nowhere else; a value near the largest number stays one."""
    def plant(q, k, v):
        q[..., 0] = 0.0
        v[40, :, 3] = float("inf")
        v[70, :, 9] = 2.0 ** 126
    assert worst_excess(((150, 400),), 4, 2, 64, 16, 1, groups, seed=6, plant=plant) <= 0.0


@pytest.mark.parametrize("hd,blocks,groups,ps,window,nsplit", [
    (64, 1, 1, 16, None, 1), (64, 1, 2, 16, None, 1), (64, 2, 2, 16, None, 1), (64, 1, 2, 16, None, 2), (128, 1, 1, 16, None, 1), (128, 1, 2, 16, None, 2),
    (64, 2, 1, 16, 700, 1), (128, 1, 1, 16, 700, 1), (64, 1, 1, 5, None, 1), (64, 2, 2, 5, None, 1), (64, 1, 1, 5, 30, 1), (48, 1, 1, 16, None, 1)])
@pytest.mark.parametrize("at", [3, 440, 860])
def test_a_key_that_is_no_number(hd, blocks, groups, ps, window, nsplit, at):
    """Every row that reads it is no number either, the others (before it, past their window, of the other key head) are what they are without it."""
    def plant(q, k, v):
        if len(k) > at:
            k[at, 0, 7] = float("nan")
    assert worst_excess(((150, 900), (60, 60), (1, 500)), 4, 2, hd, ps, blocks, groups, nsplit, window, seed=9, plant=plant) <= 0.0


@pytest.mark.parametrize("blocks,groups", [(1, 1), (2, 1), (2, 2)])
def test_a_workgroup_goes_from_a_tile_that_is_made_again_to_the_next(blocks, groups):
    assert worst_excess(((1530, 1530),), 32, 8, 64, 16, blocks, groups, seed=7, plant=planted(120.0, 1000, 701)) <= 0.0
