"""Into how many runs the float32 prompt attention cuts the keys: the rule alone."""
import pytest
import torch

from nanoinfer_amd import kernels as K


@pytest.mark.parametrize("hd,kv_heads,group", [(64, 8, 4), (128, 8, 3)])
def test_portions_beside_others_stay_in_one_run_under_512_keys(hd, kv_heads, group):
    def runs(keys, alone):
        return K.mfma_splits(9, kv_heads, group, keys, hd, torch.float32, alone)

    for keys in (100, 255):
        assert runs(keys, True) == runs(keys, False) == 1
    for keys in (256, 300, 511):
        assert runs(keys, True) > 1 and (runs(keys, False) == 1 if hd == 64 else runs(keys, False) == runs(keys, True))
    for keys in (512, 1500):
        assert runs(keys, True) == runs(keys, False) > 1


def test_how_many_runs():
    """At most sixteen and never more than there are steps of 32 keys; one where the tiles alone fill the chip for rounds."""
    for tiles in (1, 16, 127, 128, 3000):
        for keys in (256, 300, 4000, 100000):
            for hd in (32, 64, 128, 256):
                if tiles * 8 >= 1024:
                    assert K.mfma_splits(tiles, 8, 4, keys, hd, torch.float32) == 1
                    continue
                assert 2 <= K.mfma_splits(tiles, 8, 4, keys, hd, torch.float32) <= min(16, -(-keys // 32))
