"""Blocks of several (batch, kv head) pairs handed out together, longest first (block_item): every block has to run exactly once,
whatever the number of pairs per XCD and of groups, against fp32 attention on the same inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, do):
    """Causal attention and its gradients in fp32, one batch entry at a time: O, LSE, dQ, dK, dV."""
    out = [[] for _ in range(5)]
    S, rep = q.shape[1], q.shape[2] // k.shape[2]
    hidden = torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1)
    for b in range(q.shape[0]):
        qb, kb, vb, db = (t[b].float().transpose(0, 1).contiguous() for t in (q, k, v, do))
        kr, vr = kb.repeat_interleave(rep, 0), vb.repeat_interleave(rep, 0)
        s = torch.matmul(qb, kr.transpose(1, 2).contiguous()) * q.shape[3] ** -0.5
        s.masked_fill_(hidden, float("-inf"))
        lse = torch.logsumexp(s, -1)
        p = torch.exp(s - lse[..., None])
        o = torch.matmul(p, vr)
        ds = p * (torch.matmul(db, vr.transpose(1, 2).contiguous()) - (db * o).sum(-1, keepdim=True)) * q.shape[3] ** -0.5
        dk, dv = (torch.matmul(t.transpose(1, 2).contiguous(), x) for t, x in ((ds, qb), (p, db)))
        fold = lambda t: t.view(-1, rep, *t.shape[1:]).sum(1)
        for dst, x in zip(out, (o, lse, torch.matmul(ds, kr), fold(dk), fold(dv))):
            dst.append(x if x.dim() == 2 else x.transpose(0, 1))
    return [torch.stack(x) for x in out]


@pytest.mark.parametrize("D,B,Hq,Hkv,S", [
    (64, 13, 8, 8, 2300),     # 13 pairs per XCD: two groups, the last one smaller
    (64, 16, 12, 12, 1024),
    (64, 5, 12, 12, 300),     # 60 pairs: they do not divide among the XCDs
    (128, 7, 8, 8, 1400),     # one group of seven
    (128, 8, 32, 8, 1000),    # four q heads per pair
    (128, 11, 16, 8, 2100),   # groups of several sizes, two q heads per pair
    (128, 1, 8, 8, 1100),     # one pair per XCD
])
def test_every_block_runs_once(ltr, D, B, Hq, Hkv, S):
    g = torch.Generator(device="cuda").manual_seed(S)
    mk = lambda h: torch.randn(B, S, h, D, generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    ref = _reference(q, k, v, do)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o, lse = ltr.block_attention(q, [k], [v], [0], causal=True)
    o.backward(do)
    got = [o.detach(), lse] + [t.grad for t in leaves]
    # bf16 results of bf16 products: 2e-3 .. 3.1e-3 of the norm; a block left out or run twice is the whole of some rows
    for name, x, r in zip(("o", "lse", "dq", "dk", "dv"), got, ref):
        x, r = x.float(), r.float()
        tiles = lambda t: (t.transpose(1, 2) if t.dim() == 4 else t).flatten(0, 1)           # [batch * heads, rows, ...]
        for first in range(0, S, 64):
            a, b = tiles(x)[:, first:first + 64], tiles(r)[:, first:first + 64]
            err = (a - b).flatten(1).norm(dim=1) / b.flatten(1).norm(dim=1).clamp_min(1e-3)
            assert err.max() < 2e-2, (name, first, err.max().item())
