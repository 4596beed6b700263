"""Bfloat16 prompt attention with a bias, caps, windows, chunks, sinks and temperatures on the matrix cores, against 64 bits of the
same rounded numbers: sizes between the compiled ones, pages of any size, tiles past the last key, values that are infinite."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def run(T, keys, H, G, dk, dv, seed, bias=False, window=None, keep=0, chunk=None, cap=None, sink=False, temp=0.0, ps=16, rising=False, spoil=None):
    """(what the kernel gives, what plain 64 bits give), [T, H, dv]; ``rising``: every key's scores are above those before it."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(seed)
    q, k, v = torch.randn(T, H, dk, generator=g), torch.randn(keys, G, dk, generator=g), torch.randn(keys, G, dv, generator=g)
    if rising:
        q, k = q.abs(), k.abs() * torch.linspace(0.1, 3.0, keys)[:, None, None]
    if spoil is not None:
        spoil(v)
    q, k, v = (t.bfloat16() for t in (q, k, v))
    pages = (keys + ps - 1) // ps
    order = torch.randperm(pages, generator=g)
    # a page that is not this sequence's holds no numbers
    kp, vp = (torch.full((pages + 1, G, ps, n), float("nan"), dtype=torch.bfloat16) for n in (dk, dv))
    for pool, t in ((kp, k), (vp, v)):
        padded = torch.full((pages * ps, *t.shape[1:]), float("nan"), dtype=torch.bfloat16)
        padded[:keys] = t
        pool[order] = padded.view(pages, ps, G, -1).permute(0, 2, 1, 3)
    table = torch.randn(40, H, generator=g) if bias else None
    sk = torch.randn(H, generator=g) if sink else None
    dev = lambda t: None if t is None else t.cuda()          # noqa: E731
    rows = K.bias_attention_mfma_rows(dk, dv)
    hpc = min(H // G, rows)
    tiles = torch.tensor(K.build_q_tiles([0], [T], [keys], rows // hpc), dtype=torch.int32).view(-1, 4)
    pos = torch.arange(keys - T, keys, dtype=torch.int32)
    out = torch.full((T + 1, H * dv), 7.0, device="cuda", dtype=torch.bfloat16)
    K.bias_attention_mfma(dev(q.reshape(T, H * dk)), dev(kp), dev(vp), order.int().view(1, -1).cuda(), dev(tiles), dev(pos), dev(table), out[:T], H, dk ** -0.5,
                          temp, 8 if temp else 0, hpc, window, keep, 0.7, sink=dev(sk), softcap=cap, chunk=chunk)
    assert bool((out[T] == 7.0).all())
    want = torch.empty(T, H, dv, dtype=torch.float64)
    for t in range(T):
        p = keys - T + t
        seen = [j for j in range(p + 1) if (chunk is None or j // chunk == p // chunk) and (window is None or p - j < window or j < keep)]
        for h in range(H):
            s = (k[seen, h // (H // G)].double() @ q[t, h].double()) * dk ** -0.5
            if temp:
                s = s * (1.0 + temp * math.log((p + 1) // 8 + 1))
            if bias:
                s = s + table[[min(p - j, 39) for j in seen], h].double()
            if cap is not None:
                s = cap * torch.tanh(s / cap)
            w = torch.softmax(torch.cat([s, sk[h:h + 1].double()]) if sink else s, 0)[:len(seen)]
            want[t, h] = 0.7 * (w @ v[seen, h // (H // G)].double())
    return out[:T].view(T, H, dv).cpu().double(), want


@pytest.mark.parametrize("H,G,dk,dv", [(4, 1, 16, 16), (6, 2, 48, 80), (4, 2, 64, 128), (3, 1, 80, 64), (2, 1, 112, 144), (2, 2, 128, 256), (2, 1, 192, 128),
                                       (2, 1, 256, 48)])
@pytest.mark.parametrize("form", [{}, {"bias": True, "temp": 0.1}, {"window": 20, "keep": 3, "sink": True}, {"chunk": 24, "cap": 3.0},
                                  {"rising": True}, {"bias": True, "cap": 20.0}])
def test_sizes_and_forms(H, G, dk, dv, form):
    for T, keys, ps in ((37, 165, 16), (20, 20, 12), (33, 64, 1), (9, 130, 7)):
        got, want = run(T, keys, H, G, dk, dv, dk + dv + T, ps=ps, **form)
        # the result's rounding; a weight is off by 2^-16 of itself and by what 2^-24 (dk + 8) of its score's products do to it,
        # scores of up to 32 and values of up to 5
        bound = 2.0 ** -8 * want.abs() + 5 * (2.0 ** -15 + 32 * 2.0 ** -24 * (dk + 8))
        assert bool(((got - want).abs() <= bound).all()), (T, keys, ps, float((got - want).abs().max()))


def test_values_that_are_not_finite():
    def spoil(v):
        v[2, 0, 5], v[3, 0, 6], v[4, 0, 7] = float("inf"), float("-inf"), float("nan")
    got, want = run(21, 130, 4, 2, 64, 64, 3, spoil=spoil)
    assert bool(got[:, :2, 7].isnan().all())
    others = [c for c in range(64) if c not in (5, 6, 7)]
    for part, full in ((got[:, :, others], want[:, :, others]), (got[:, 2:], want[:, 2:])):
        assert bool(((part - full).abs() <= 2.0 ** -8 * full.abs() + 1e-3).all())
    assert not bool(torch.isfinite(got[:, :2, 5:7]).any())
