"""Float32 attention of single tokens by 4 x 4 blocks: groups of query heads about the four that fit, contexts about a step
of sixteen keys, windows, and page sizes that are no power of two."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,group,KVH,PS", [(16, 1, 2, 16), (64, 3, 2, 12), (64, 4, 1, 16), (128, 3, 2, 16), (48, 2, 3, 5), (256, 4, 1, 16),
                                             (64, 5, 1, 16), (80, 17, 1, 8)])
@pytest.mark.parametrize("window,runs", [(None, 1), (None, 3), (21, 1), (100, 2)])
def test_few_heads(hd, group, KVH, PS, window, runs):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(hd * group + runs)
    lengths = [1, 15, 16, 17, 64, 65, 130, 700]
    T, H = len(lengths), group * KVH
    need = [(n + PS - 1) // PS for n in lengths]
    order = torch.randperm(sum(need), generator=g).int()
    table, at = torch.full((T, max(need)), -1, dtype=torch.int32), 0
    for t, n in enumerate(need):
        table[t, :n] = order[at:at + n]
        at += n
    q = torch.randn(T, (H + 2 * KVH) * hd, generator=g)
    q[3] *= 30.0                                     # scores that rise far above the first reference
    kp, vp = (torch.randn(sum(need), KVH, PS, hd, generator=g) for _ in range(2))
    out, ws = torch.full((T + 1, H * hd), 7.0, device="cuda"), torch.full((T * H * runs * (hd + 2),), float("nan"), device="cuda")
    K.mfma_token_attention(q.cuda(), kp.cuda(), vp.cuda(), table.cuda(), torch.arange(T, dtype=torch.int32, device="cuda"),
                           torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device="cuda"), out[:T], H, KVH, hd, hd ** -0.5,
                           window, runs, ws)
    assert bool((out[T] == 7.0).all())
    for t, n in enumerate(lengths):
        k, v = (p[table[t, :need[t]].long()].permute(1, 0, 2, 3).reshape(KVH, -1, hd)[:, max(0, n - (window or n)):n].double() for p in (kp, vp))
        qt = q[t, :H * hd].double().view(KVH, group, hd)
        s = qt @ k.transpose(1, 2) * hd ** -0.5
        want = (torch.softmax(s, dim=-1) @ v).reshape(-1)
        # a score's error moves a weight by as much of itself: hd + 4 roundings of the score's terms; and one per key of the sums
        size = (qt.abs() @ k.abs().transpose(1, 2)).max().item() * hd ** -0.5
        bound = 2.0 ** -24 * (2 * (hd + 4) * size + n + 64) * v.abs().max().item()
        assert float((out[t].double().cpu() - want).abs().max()) <= bound, (t, n)
