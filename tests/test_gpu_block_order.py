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
    (96, 13, 8, 8, 2300),     # padded head dims: groups of 7 + 6 and 5 + 5 + 3 pairs, places of the last one empty
    (40, 13, 8, 8, 2300),
    (128, 5, 8, 8, 2500),     # 3 + 2
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


@pytest.mark.parametrize("B,H", [(65536, 8), (65537, 8)])   # no empty place in the last group; one per XCD
def test_more_pairs_than_places_of_the_grid(ltr, B, H):
    """65536 pairs per XCD: one more than the grid's third dimension holds.  Two rows and keys, against the closed form."""
    g = torch.Generator(device="cuda").manual_seed(B)
    q, k, v, do = (torch.randn(B, 2, H, 64, generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o, lse = ltr.block_attention(q, [k], [v], [0], causal=True)
    o.backward(do)
    qf, kf, vf, df = (t.detach().float() for t in (q, k, v, do))
    s = torch.stack([(qf[:, 1] * kf[:, j]).sum(-1) for j in range(2)], -1) / 8         # row 1: [B, H, 2]; row 0 sees key 0 alone
    p = torch.softmax(s, -1)
    o1 = p[..., :1] * vf[:, 0] + p[..., 1:] * vf[:, 1]
    dp = torch.stack([(df[:, 1] * vf[:, j]).sum(-1) for j in range(2)], -1)
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) / 8
    ref = {"o": torch.stack([vf[:, 0], o1], 1), "dq": torch.stack([torch.zeros_like(o1), ds[..., :1] * kf[:, 0] + ds[..., 1:] * kf[:, 1]], 1),
           "dk": torch.stack([ds[..., j:j + 1] * qf[:, 1] for j in range(2)], 1),
           "dv": torch.stack([df[:, 0] + p[..., :1] * df[:, 1], p[..., 1:] * df[:, 1]], 1)}
    assert (lse[:, :, 1] - torch.logsumexp(s, -1)).abs().max() < 2e-2
    # bf16 operands and results: 3e-3 of a row's norm, 2e-2 with the largest of a million rows.  dS = P (dO . v - DELTA) besides has DELTA from
    # the bf16 O: 64 products of order 1 rounded to 2^-9 each, 0.016 rms and 0.1 at six sigma, times |k| / 8 of at most 1.5 (dQ; dK alike).
    # A block left out or run twice is the whole of a row, of norm 3 .. 10
    for name, got in (("o", o.detach()), ("dq", q.grad), ("dk", k.grad), ("dv", v.grad)):
        err, norm = (got.float() - ref[name]).flatten(2).norm(dim=2) / H ** 0.5, ref[name].flatten(2).norm(dim=2) / H ** 0.5
        assert (err <= 2e-2 * norm + 0.15).all(), (name, (err - 2e-2 * norm).max().item())
