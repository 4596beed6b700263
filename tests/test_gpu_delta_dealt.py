"""The delta rule in runs of sixteen: a sequence's workgroups are dealt to all dies, whatever the number of sequences; every sequence gets what it
gets alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 3, 4, 6, 8, 12, 16, 20, 24])
def test_every_sequence_is_walked_once_and_as_alone(B):
    from nanoinfer_amd import kernels as K
    g = torch.Generator().manual_seed(B)
    G, H, dk, dv, taps = 1, 5, 32, 40, 4
    lens = [1 + (7 * i) % 5 for i in range(B)]
    lens[B // 2] = 130
    starts = [sum(lens[:i]) for i in range(B)]
    T, C = sum(lens), 2 * G * dk + H * dv
    rand = lambda *s: torch.randn(*s, generator=g).cuda()                    # noqa: E731
    proj, low, conv = rand(T, C + H), rand(T, H * dk + H * dv), rand(C, taps) * 0.7
    a_log, dt_bias, norm_w = rand(H) * 0.3 - 1.0, rand(H * dk), rand(dv)
    state = rand(B, H * dv * dk + (taps - 1) * C) * 0.5
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")        # noqa: E731

    def run(which, st):
        rows = torch.cat([torch.arange(starts[s], starts[s] + lens[s]) for s in which]).cuda()
        mine = [lens[s] for s in which]
        return K.delta_rule(proj[rows].contiguous(), low[rows].contiguous(), conv, a_log, dt_bias, norm_w, st,
                            i32([i for i, n in enumerate(mine) for _ in range(n)]), i32([sum(mine[:i]) for i in range(len(mine))]), i32(mine), i32(list(which)),
                            G, H, dk, dv, taps, 1e-5, torch.float32, max_q_len=max(mine), runs=True)

    together, states = state.clone(), state.clone()
    got = run(range(B), together)
    for s in range(B):
        assert torch.equal(got[starts[s]:starts[s] + lens[s]], run([s], states)), s
    assert torch.equal(together, states)
