"""Portions that are alone in their step: the kernels of the short convolutions then move the tails on themselves.  Outputs and tails are those of
the same rows beside another sequence, whose tails a launch behind moves, bit for bit."""
from types import SimpleNamespace

import pytest
import torch

from nanoinfer_amd import kernels as K

pytestmark = pytest.mark.gpu


def _step(lens, slots):
    dev = torch.device("cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)      # noqa: E731
    starts = [sum(lens[:i]) for i in range(len(lens))]
    seq = SimpleNamespace(q_start=i32(starts), q_len=i32(lens), context_len=i32(lens), state_slot=i32(slots))
    return SimpleNamespace(seq_of_token=i32([b for b, n in enumerate(lens) for _ in range(n)]), per_seq=seq, max_q_len=max(lens), i32=i32)


def _noise(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator("cpu").manual_seed(seed)).cuda()


@pytest.mark.parametrize("taps", [2, 4, 5, 7])
@pytest.mark.parametrize("T", [2, 5, 63, 64, 66, 257])
@pytest.mark.parametrize("d,dtype", [(96, torch.bfloat16), (50, torch.float32), (128, torch.float32)])
def test_input_convolution(T, taps, d, dtype):
    h, w, state = _noise(1, T + 2, d), _noise(2, d, taps), _noise(3, 3, 8 + (taps - 1) * d)
    got = {}
    for lens in ([T], [T, 2]):
        st, rows = state.clone(), sum(lens)
        x = torch.empty(rows, d, dtype=dtype, device="cuda")
        K.input_conv(h[:rows].contiguous(), K.InputConv(w, st, 8, _step(lens, [1, 2][:len(lens)])), x)
        got[len(lens)] = x[:T], st[1], st[0]
    for a, b in zip(got[1], got[2]):
        assert torch.equal(a, b)
    tail = torch.cat([state[1, 8:].view(taps - 1, d), h[:T]])[-(taps - 1):]
    assert torch.equal(got[1][1][8:].view(taps - 1, d), tail)


@pytest.mark.parametrize("T", [2, 9, 63, 64, 65, 300])
@pytest.mark.parametrize("taps,H,G,maps,dk,dv", [(4, 4, 2, 2, 64, 128), (4, 3, 1, 1, 128, 96), (4, 2, 2, 1, 192, 256), (4, 2, 1, 1, 33, 40), (3, 2, 1, 1, 64, 64)])
def test_projected_queries_keys_and_values(T, taps, H, G, maps, dk, dv):
    C, ps = (H + G) * maps * dk + G * dv, 16
    proj, w, state = _noise(4, T + 1, C + 6), _noise(5, C, taps), _noise(6, 3, (taps - 1) * C)
    got = {}
    for lens in ([T], [T, 1]):
        st, rows, pages = state.clone(), sum(lens), T // ps + 2
        ctx = _step(lens, [1, 2][:len(lens)])
        kpool, vpool = (torch.zeros(pages, G, ps, n, dtype=torch.bfloat16, device="cuda") for n in (maps * dk, dv))
        q = torch.empty(rows, H * maps * dk, dtype=torch.bfloat16, device="cuda")
        K.qkv_conv(proj[:rows].contiguous(), ctx.i32(list(range(T)) + [0][:rows - T]), ctx.i32(list(range(T)) + [(pages - 1) * ps][:rows - T]), w, None, None, 1e-6,
                   None, st, 0, ctx, q, kpool, vpool, H, maps)
        got[len(lens)] = q[:T], st[1], st[0], kpool[:-1], vpool[:-1]
    for a, b in zip(got[1], got[2]):
        assert torch.equal(a, b)
    tail = torch.cat([state[1].view(taps - 1, C), proj[:T, :C]])[-(taps - 1):]
    assert torch.equal(got[1][1].view(taps - 1, C), tail)
