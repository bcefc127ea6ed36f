"""CPU tests of which way the context-parallel layer takes: the shards as one sequence, or one launch per shard."""
from types import SimpleNamespace

import pytest
import torch

import lightron_amd as la


def _choice(W, B, n, H, Hkv, D, train, causal=True):
    args = SimpleNamespace(dim=H * D, n_heads=H, n_kv_heads=Hkv, tp_size=1)
    with torch.device("meta"):
        layer = la.ContextParallelAttention(la.Attention(args).to(torch.bfloat16), args, cp_group=la.LocalCPGroup(W), causal=causal)
        x = torch.empty(W, B, n, H * D, dtype=torch.bfloat16)
    with torch.set_grad_enabled(train):
        return layer._one_sequence(x, W * n)


@pytest.mark.parametrize("causal", [True, False])
def test_one_batch_entry_and_training_take_the_sequence(causal):
    for W, B, n, H in ((2, 1, 37, 8), (4, 1, 8192, 32), (2, 16, 2048, 16), (4, 8, 128, 32)):
        assert _choice(W, B, n, H, H, 128, True, causal)
        assert _choice(W, B, n, H, H, 128, False, causal) == (B == 1 or n == 128)


def test_forward_only_joins_shards_where_it_saves_more_than_its_copies():
    assert not _choice(2, 8, 1024, 16, 16, 128, False)
    assert not _choice(2, 8, 1024, 16, 4, 64, False)
    assert _choice(4, 16, 128, 16, 4, 64, False)           # launches cost more than the copies
    assert _choice(2, 8, 2048, 12, 12, 64, False)          # a shard's launch leaves CUs idle, the sequence's does not
    assert _choice(2, 8, 512, 16, 16, 128, False, causal=False) is False


def test_sequences_past_the_kernels_limits_stay_shards():
    """The dK/dV kernel lists at most 4096 q tiles of 64 rows; tile offsets inside a chunk are 32-bit element counts."""
    assert _choice(2, 1, 131072, 2, 2, 64, True)
    assert not _choice(2, 1, 131104, 2, 2, 64, True)
    assert _choice(2, 1, 131104, 2, 2, 64, False)
    assert not _choice(4, 1, 131072, 32, 8, 128, False)
    assert not _choice(8, 1, 65536, 32, 32, 128, True)
