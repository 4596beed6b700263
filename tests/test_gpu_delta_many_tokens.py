"""The delta rule over many tokens of many short and some longer sequences."""
import pytest
import torch

from test_gpu_zekalorn import _plain_delta_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,H,dk,dv,taps", [(1, 2, 32, 24, 4), (1, 1, 16, 130, 4), (2, 2, 80, 16, 4), (1, 1, 128, 64, 4), (1, 2, 48, 16, 3), (1, 1, 144, 20, 1)])
def test_many_tokens_agree_with_the_plain_recurrence(G, H, dk, dv, taps):
    """Sequences that begin and end within four tokens, on their filters' first inputs and far behind them."""
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(dk + dv)
    lens = [2, 5, 70, 1, 3, 130, 4, 48]
    starts = [sum(lens[:i]) for i in range(len(lens))]
    slots = [3, 0, 4, 1, 6, 2, 8, 7]
    T, C = sum(lens), 2 * G * dk + H * dv
    assert T > 256 and T % 4
    rand = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)      # noqa: E731
    proj, low, conv = rand(T, C + H) * 1.5, rand(T, H * dk + H * dv), rand(C, taps) * 0.7
    a_log, dt_bias, norm_w = rand(H) * 0.3 - 1.0, rand(H * dk), torch.rand(dv, generator=g, dtype=torch.float64) + 0.5
    state = rand(9, H * dv * dk + (taps - 1) * C) * 0.5
    want, want_state = _plain_delta_step(proj, low, conv, a_log, dt_bias, norm_w, state, starts, lens, slots, G, H, dk, dv, taps, 1e-5)
    f32 = lambda t: t.to("cuda", torch.float32).contiguous()                 # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")        # noqa: E731
    seq_of_token = i32([s for s, n in enumerate(lens) for _ in range(n)])
    for runs in (True, False):
        st = f32(state)
        got = K.delta_rule(f32(proj), f32(low), f32(conv), f32(a_log), f32(dt_bias), f32(norm_w), st, seq_of_token, i32(starts), i32(lens), i32(slots),
                           G, H, dk, dv, taps, 1e-5, torch.float32, max_q_len=max(lens), runs=runs)
        # the bound that steps of fewer tokens are held to
        assert float((got.double().cpu() - want).abs().max() / want.abs().max()) < 2e-5, runs
        assert float((st.double().cpu() - want_state).abs().max() / want_state.abs().max()) < 2e-5, runs
