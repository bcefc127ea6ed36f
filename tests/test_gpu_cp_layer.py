"""The context-parallel layer's two ways through the attention (shards as one sequence, one launch per shard), on the GPU."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(ltr, W, H, Hkv, D, dtype, **kw):
    g = torch.Generator(device="cuda").manual_seed(H + D)
    args = SimpleNamespace(dim=H * D, n_heads=H, n_kv_heads=Hkv, tp_size=1)
    with torch.device("cuda"):
        inner = ltr.Attention(args).to(dtype)
    for p in inner.parameters():
        p.data.normal_(0, (H * D) ** -0.5, generator=g)
    return ltr.ContextParallelAttention(inner, args, cp_group=ltr.LocalCPGroup(W), **kw), g


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.parametrize("W,B,n,H,Hkv,D,dtype,causal", [
    (2, 3, 77, 4, 2, 64, torch.bfloat16, True),
    (4, 2, 130, 8, 8, 128, torch.bfloat16, False),
    (2, 2, 65, 2, 2, 64, torch.float32, True),
])
def test_both_ways_agree(ltr, W, B, n, H, Hkv, D, dtype, causal, monkeypatch):
    layer, g = _layer(ltr, W, H, Hkv, D, dtype, causal=causal)
    freqs = ltr.precompute_freqs_cis(D, W * n, device="cuda")
    x, do = (torch.randn(W, B, n, H * D, device="cuda", dtype=dtype, generator=g) for _ in range(2))
    res = []
    for one in (True, False):
        monkeypatch.setattr(layer, "_one_sequence", lambda *a, one=one: one)
        xl = x.clone().requires_grad_(True)
        y = layer(xl, freqs)
        assert y.is_contiguous() and y.shape == x.shape
        y.backward(do)
        res.append([y.detach(), xl.grad] + [p.grad for p in layer.parameters()])
        for p in layer.parameters():
            p.grad = None
    # the same values but for the order of fp32 sums (and, per shard, dK / dV rounded to bf16 before they are added)
    for a, b in zip(*res):
        assert _rel(a, b) < (1e-2 if dtype == torch.bfloat16 else 1e-5)


def test_sequence_longer_than_one_backward_launch(ltr):
    """262208 tokens: more than the 4096 q tiles that a backward launch lists; the shards are attended one by one."""
    W, n, H, D = 2, 131104, 2, 64
    layer, g = _layer(ltr, W, H, H, D, torch.bfloat16)
    freqs = ltr.precompute_freqs_cis(D, W * n, device="cuda")
    x = torch.randn(W, 1, n, H * D, device="cuda", dtype=torch.bfloat16, generator=g).requires_grad_(True)
    y = layer(x, freqs)
    y.backward(torch.randn(y.shape, device="cuda", dtype=y.dtype, generator=g))
    assert torch.isfinite(x.grad).all() and x.grad.float().norm() > 0
    with torch.no_grad():       # forward only, the whole is one sequence
        assert _rel(y.detach(), layer(x, freqs)) < 1e-2
