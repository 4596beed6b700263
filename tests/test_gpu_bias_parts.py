"""Float32 prompt attention with a bias, caps, windows, chunks, maps, sinks and gates in three bfloat16 parts, against 64 bits: sizes
between the compiled ones, and numbers that are not finite or too large for a bfloat16."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def run(T, keys, H, G, dk, dv, seed, bias=False, window=None, keep=0, chunk=None, cap=None, sink=False, gate=False, temp=0.0, spoil=None, ps=16):
    """(what the kernel gives, what plain 64 bits give), [T, H, dv]."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(seed)
    q, k, v = torch.randn(T, H, dk, generator=g), torch.randn(keys, G, dk, generator=g), torch.randn(keys, G, dv, generator=g)
    if spoil is not None:
        spoil(q, k, v)
    pages = (keys + ps - 1) // ps
    order = torch.randperm(pages, generator=g)
    kp, vp = torch.zeros(pages, G, ps, dk), torch.zeros(pages, G, ps, dv)
    for pool, t in ((kp, k), (vp, v)):
        padded = torch.zeros(pages * ps, *t.shape[1:])
        padded[:keys] = t
        pool[order] = padded.view(pages, ps, G, -1).permute(0, 2, 1, 3)
    table = torch.randn(40, H, generator=g) if bias else None
    sk = torch.randn(H, generator=g) if sink else None
    rows = torch.randn(T, H * dv, generator=g) if gate else None
    dev = lambda t: None if t is None else t.cuda()          # noqa: E731
    hpc = min(H // G, K.bias_attention_mfma_rows(dk, dv))
    tiles = torch.tensor(K.build_q_tiles([0], [T], [keys], K.bias_attention_mfma_rows(dk, dv) // hpc), dtype=torch.int32).view(-1, 4)
    pos = torch.arange(keys - T, keys, dtype=torch.int32)
    out = torch.empty(T, H * dv, device="cuda")
    K.bias_attention_mfma(dev(q.reshape(T, H * dk)), dev(kp), dev(vp), order.int().view(1, -1).cuda(), dev(tiles), dev(pos), dev(table), out, H, dk ** -0.5,
                          temp, 8 if temp else 0, hpc, window, keep, 0.7, sink=dev(sk), softcap=cap, chunk=chunk,
                          gate=None if rows is None else (dev(rows), 0, 1))
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
    if gate:
        want = want * torch.sigmoid(rows.double()).view(T, H, dv)
    return out.view(T, H, dv).cpu(), want


@pytest.mark.parametrize("H,G,dk,dv", [(4, 1, 16, 16), (6, 2, 48, 80), (4, 2, 64, 128), (3, 1, 80, 64), (2, 1, 112, 144), (2, 2, 128, 256), (2, 1, 144, 64)])
@pytest.mark.parametrize("form", [{}, {"bias": True, "temp": 0.1}, {"window": 20, "keep": 3, "sink": True}, {"chunk": 24, "cap": 3.0}, {"gate": True, "bias": True, "cap": 20.0}])
def test_sizes_and_forms(H, G, dk, dv, form):
    for T, keys, ps in ((37, 101, 16), (20, 20, 12), (33, 64, 8)):
        got, want = run(T, keys, H, G, dk, dv, dk + dv + T, ps=ps, **form)
        # scores of up to 5 sums of dk products, 2^-24 (dk + 6) of their terms' size each, move a weight by as much of itself
        assert float((got.double() - want).abs().max()) <= 2.0 ** -24 * (8 * (dk + 6) + keys) * 4.0, (T, keys)


@pytest.mark.parametrize("dk,dv", [(64, 64), (32, 128), (128, 64)])
def test_what_is_not_finite_or_too_large(dk, dv):
    def values(q, k, v):
        v[2, 0, 5], v[3, 0, 6], v[4, 0, 7], v[5, 0, 8] = float("inf"), float("-inf"), float("nan"), 3.4e38
    got, want = run(21, 60, 4, 2, dk, dv, 3, spoil=values)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got) * torch.sign(got), torch.isinf(want) * torch.sign(want).float())
    fine = torch.isfinite(want)
    assert float(((got.double() - want) / want.abs().clamp(min=1.0))[fine].abs().max()) <= 1e-5

    def keys(q, k, v):      # a key that is the only one or none
        q[:, :, 9] = torch.where(q[:, :, 9] < 0, -0.02, 0.02)
        k[1] = 0.0
        k[1, :, 9] = 3.4e38
    got, want = run(21, 60, 4, 2, dk, dv, 4, spoil=keys)
    assert float((got.double() - want).abs().max()) <= 1e-5
