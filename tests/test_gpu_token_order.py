"""Single tokens on the matrix cores, uncut: each workgroup finds its token by the order of the positions.  Whatever order the
tokens come in, every one gets bit for bit what it gets alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("T,H,KVH,order", [(2, 4, 2, "rising"), (3, 6, 3, "mixed"), (33, 8, 4, "mixed"), (64, 32, 8, "mixed"), (64, 16, 8, "equal"),
                                           (63, 16, 8, "falling"), (256, 4, 2, "mixed"), (257, 4, 2, "mixed"), (129, 8, 4, "mixed")])
def test_tokens_in_any_order(dtype, hd, T, H, KVH, order):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(T)
    length = torch.randint(1, 150, (T,), generator=g)
    if order == "equal":
        length[:] = 77
    elif order != "mixed":
        length = torch.sort(length, descending=order == "falling").values
    pages = int(((length + 15) // 16).sum())
    place = torch.randperm(pages, generator=g)
    table = torch.full((T, 10), -1, dtype=torch.int32)
    at = 0
    for t in range(T):
        n = int(length[t] + 15) // 16
        table[t, :n] = place[at:at + n]
        at += n
    k, v = (torch.randn(pages, KVH, 16, hd, generator=g).cuda().to(dtype) for _ in range(2))
    q = torch.randn(T, (H + 2 * KVH) * hd, generator=g).cuda().to(dtype)
    positions, table, seq = (length - 1).int().cuda(), table.cuda(), torch.arange(T, dtype=torch.int32).cuda()

    def attend(rows):
        out = torch.full((len(rows), H * hd), float("nan"), device="cuda", dtype=dtype)
        return K.mfma_token_attention(q[rows].contiguous(), k, v, table, seq[rows].contiguous(), positions[rows].contiguous(), out, H, KVH, hd,
                                      hd ** -0.5, None, 1)
    together = attend(list(range(T)))
    for t in list(range(min(T, 40))) + [T - 1]:
        assert torch.equal(together[t], attend([t])[0]), t
    swapped = list(reversed(range(T)))
    assert torch.equal(attend(swapped), together[swapped])
