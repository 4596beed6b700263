"""The delta rule over sequences of as many runs of sixteen as the chain holds ahead, of fewer and of more, and over steps whose rows
are prepared four tokens at a time (448 tokens and more, 64 a sequence)."""
import pytest
import torch

from test_gpu_zekalorn import _plain_delta_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1, 16, 17, 31, 32, 33, 47, 48], [49, 64, 1, 65, 80, 2, 81, 97],       # one run, two, three and more
                                  [2, 5, 70, 1, 3, 330, 4, 200], [448], [3, 509]])                       # four tokens at a time
@pytest.mark.parametrize("G,H,dk,dv,taps", [(1, 2, 32, 24, 4), (1, 1, 96, 40, 4), (1, 1, 128, 64, 4), (1, 1, 80, 16, 3), (1, 1, 144, 20, 1)])
def test_runs_held_ahead(lens, G, H, dk, dv, taps):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(dk + dv + len(lens))
    starts = [sum(lens[:i]) for i in range(len(lens))]
    slots = [3, 0, 4, 1, 6, 2, 8, 7][:len(lens)]
    T, C = sum(lens), 2 * G * dk + H * dv
    rand = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)      # noqa: E731
    proj, low, conv = rand(T, C + H) * 1.5, rand(T, H * dk + H * dv), rand(C, taps) * 0.7
    a_log, dt_bias, norm_w = rand(H) * 0.3 - 1.0, rand(H * dk), torch.rand(dv, generator=g, dtype=torch.float64) + 0.5
    state = rand(9, H * dv * dk + (taps - 1) * C) * 0.5
    want, want_state = _plain_delta_step(proj, low, conv, a_log, dt_bias, norm_w, state, starts, lens, slots, G, H, dk, dv, taps, 1e-5)
    f32 = lambda t: t.to("cuda", torch.float32).contiguous()                 # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")        # noqa: E731
    st = f32(state)
    got = K.delta_rule(f32(proj), f32(low), f32(conv), f32(a_log), f32(dt_bias), f32(norm_w), st, i32([s for s, n in enumerate(lens) for _ in range(n)]),
                       i32(starts), i32(lens), i32(slots), G, H, dk, dv, taps, 1e-5, torch.float32, max_q_len=max(lens), runs=True)
    # the bound that the delta rule's other tests hold it to
    assert float((got.double().cpu() - want).abs().max() / want.abs().max()) < 2e-5
    assert float((st.double().cpu() - want_state).abs().max() / want_state.abs().max()) < 2e-5
