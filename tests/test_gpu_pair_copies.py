"""The copy of large float32 matrices as pairs of halves: made where it leaves as much device memory as it takes, never in the way of
a model that only fits without it, and switched off by itself."""
import pytest
import torch

from test_gpu_parts import random_tensors

pytestmark = pytest.mark.gpu

CONFIG = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": 1024, "num_hidden_layers": 2, "num_attention_heads": 16,
          "num_key_value_heads": 4, "head_dim": 64, "intermediate_size": 4096, "vocab_size": 512, "rms_norm_eps": 1e-5, "rope_theta": 500000.0,
          "max_position_embeddings": 2048, "tie_word_embeddings": False, "hidden_act": "silu"}
MATRICES = 2 * 1024 * (1024 + 512 + 1024 + 2 * 4096 + 4096)          # numbers in the layers' matrices


def runner(monkeypatch, free=None, **options):
    from nanoinfer_amd.engine import runner as R
    from nanoinfer_amd.registry import architecture_of
    arch = architecture_of(CONFIG)
    spec = arch.build_spec(arch.config_from_dict(CONFIG))
    if free is not None:
        monkeypatch.setattr(R._Gpu, "free_bytes", staticmethod(lambda: free))
    return R.ModelRunner.from_spec(spec, random_tensors(spec, 3), dtype="float32", max_tokens=1024, max_requests=2, **options)


def prompt(r):
    from nanoinfer_amd.engine.runner import StepEntry
    tokens = torch.randint(0, 512, (600,), generator=torch.Generator().manual_seed(2)).tolist()
    return r.step([StepEntry("p", tokens, [599])], end=["p"]).double()


def held(r):
    return sum(w.pairs is not None for w in r.rt._for_pairs)


def test_the_copy_is_made_where_it_leaves_as_much_as_it_takes(monkeypatch):
    full = runner(monkeypatch)
    need = sum(w.pair_bytes() for w in full.rt._for_pairs)
    assert held(full) == 8 and 4 * MATRICES <= need <= 4.1 * MATRICES
    want = prompt(full)
    bytes_of = full.memory_report()["weights"]
    for tight in (runner(monkeypatch, free=2 * need - 1), runner(monkeypatch, pair_copies=False), runner(monkeypatch, free=0)):
        assert held(tight) == 0 and tight.memory_report()["weights"] == bytes_of - need
        assert float((prompt(tight) - want).norm() / want.norm()) <= 2e-5          # the products in three parts
    assert held(runner(monkeypatch, free=2 * need)) == 8
    assert held(runner(monkeypatch, one_weight_copy=True)) == 0


def test_bytes_of_the_copy():
    from nanoinfer_amd import kernels as K
    for N, Kd in ((512, 1024), (513, 1028), (4096, 132)):
        w = K.Weight(torch.randn(N, Kd, device="cuda"))
        assert w.pair_bytes() == sum(t.numel() * t.element_size() for t in w.pairs) == K.pair_weight_bytes(N, Kd)
    assert K.Weight(torch.randn(512, 1026, device="cuda")).pair_bytes() == 0
