"""bwd_joint_kernel (dQ and dK/dV blocks in one launch) against the dense oracle and against the two launches it takes the place of, at the
edges of both kinds' tiles (128 or 256 rows, 64-row sub-tiles, 128 keys), dQ blocks first and dK/dV blocks first."""
import pytest
import torch

from attn_abi import backward
from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


DQ_FIRST = [
    (64, 2, 12, 12, 1, 0, None, [(1, 0)], True),                                   # one row, one key
    (64, 4, 12, 12, 128, 0, None, [(128, 0)], True),
    (64, 1, 8, 2, 321, 0, None, [(321, 0)], True),                                 # grouped heads, pairs that do not divide among the XCDs
    (64, 3, 16, 16, 193, (40, 300), 33, [(31, 0), (130, 31), (64, 500)], True),    # two segments, chunk tails, keys no row sees
    (64, 2, 16, 8, 160, 5, None, [(165, 0)], True),                                # DELTA by the blocks: 2 heads x 160 rows, their most
    (128, 1, 16, 16, 144, 0, None, [(144, 0)], True),                              # one head of 144
    (128, 2, 8, 8, 97, 0, None, [(97, 0)], False),
    (120, 1, 8, 8, 101, 0, None, [(101, 0)], True),
    (128, 2, 8, 8, 257, 0, None, [(257, 0)], True),                                # one row and key past two tiles
    (128, 1, 32, 8, 700, 0, None, [(700, 0)], True),                               # shared key tiles
    (128, 1, 16, 16, 500, 37, None, [(300, 0), (129, 300)], False),
    (128, 5, 8, 8, 450, 0, None, [(450, 0)], True),
    (128, 5, 32, 32, 240, 0, None, [(240, 0)], False),                             # more blocks than CUs
    (96, 2, 16, 16, 391, 0, None, [(391, 0)], True),
    (40, 1, 8, 4, 130, 3, None, [(133, 0)], True),
]
ZIGZAG = lambda h: [(h, 0), (h, h), (h, 2 * h), (h, 3 * h)]
KEYS_FIRST = [
    (64, 5, 48, 12, 110, 0, None, [(110, 0)], True),                               # pairs that do not divide among the XCDs
    (64, 3, 64, 16, 72, (36, 72), 36, ZIGZAG(36), True),                           # grouped block order, keys no row sees
    (64, 2, 128, 32, 134, 0, None, [(134, 0)], True),                              # 256-row dQ blocks
    (64, 3, 32, 8, 265, 0, None, [(265, 0)], True),                                # shared key tiles
    (128, 5, 16, 8, 264, 0, None, [(264, 0)], True),
    (128, 5, 48, 12, 132, 0, None, [(132, 0)], True),
    (128, 3, 32, 8, 271, 0, None, [(271, 0)], True),                               # shared key tiles
    (128, 5, 32, 8, 90, (45, 90), 45, ZIGZAG(45), True),
    (96, 3, 64, 32, 112, 0, None, [(112, 0)], False),
    (120, 5, 32, 8, 66, (33, 66), 33, ZIGZAG(33), True),
    (40, 5, 16, 4, 307, 0, None, [(307, 0)], False),
]


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,split,chunks,causal,keys_first", [(*c, False) for c in DQ_FIRST] + [(*c, True) for c in KEYS_FIRST])
def test_joint(ltr, D, B, Hq, Hkv, Sq, q_pos, split, chunks, causal, keys_first):
    """bf16 results with DELTA from o, and fp32 accumulators with DELTA given: each in the joint launch that its own plan names, in this order."""
    total, pos = sum(n for n, _ in chunks), [p for _, p in chunks]
    g = torch.Generator().manual_seed(Sq)
    mk = lambda s, h: torch.randn(B, s, h, D, generator=g).to(torch.bfloat16)
    q, do, k, v = mk(Sq, Hq), mk(Sq, Hq), mk(total, Hkv), mk(total, Hkv)
    at = [sum(n for n, _ in chunks[:i]) for i in range(len(chunks))]
    cut = lambda t: [t[:, a:a + n] for a, (n, _) in zip(at, chunks)]
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    rows = torch.arange(Sq)
    qpos = rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    _, _, *ref = orc.dense_attention_grads(q.float(), k.float(), v.float(), do.float(), qpos, kpos, causal, dtype=torch.float32)
    qd, kd, vd, dod = q.cuda(), k.cuda(), v.cuda(), do.cuda()
    o, lse = (t.detach() for t in ltr.block_attention(qd, cut(kd), cut(vd), pos, q_pos, split, causal))

    def run(joint, results, fill, delta=None):
        got = backward(qd, dod, o, lse, cut(kd), cut(vd), pos, q_pos, split, causal, joint, results, fill, delta)
        pad = "" if D in (64, 128) else "_pad"
        names = {"bwd_joint%s_kernel<%d, %d>" % (pad, 64 if D <= 64 else 128, 256 // got.plan.rows)}
        if delta is None:
            names.add("bwd_joint_delta%s_kernel<%d>" % (pad, 64 if D <= 64 else 128))
        assert (got.plan.dq in names and got.plan.dkdv == got.plan.dq) if joint else not names & {got.plan.dq, got.plan.dkdv}
        assert got.plan.keys_first == (joint and keys_first)
        return got

    # bf16 P, dS, products and results: 2e-3 .. 3.1e-3 of the norm.  With one key dS = dP - DELTA is zero but for the rounding of two fp32 sums of
    # size 8 (1e-6), times a key and 1 / sqrt(D): 1e-6 per element.  Results where no query sees a key are zeros
    direct = run(True, torch.bfloat16, 7.0)
    for name, want in zip(("dq", "dk", "dv"), ref):
        assert (getattr(direct, name).cpu().float() - want).norm() <= 1e-2 * want.norm() + 1e-6 * want.numel() ** 0.5, name
    seen = torch.ones(total, dtype=torch.bool) if not causal else kpos <= qpos.max()
    assert not direct.dk.cpu()[:, ~seen].any() and not direct.dv.cpu()[:, ~seen].any()
    want_delta = (do.float() * o.cpu().float()).sum(-1).transpose(1, 2)
    assert (direct.delta.cpu() - want_delta).abs().max() <= 1e-5 * D + 1e-5 * want_delta.abs().max()
    again = run(True, torch.bfloat16, 7.0)
    assert all(torch.equal(getattr(direct, n), getattr(again, n)) for n in ("dq", "dk", "dv", "delta"))
    # fp32 accumulators with DELTA given: the sums of the two launches in another order, added to what was there
    delta = ltr.attn_delta(o, dod)
    joint, apart = (run(j, torch.float32, 0.5, delta) for j in (True, False))
    for name, want in zip(("dq", "dk", "dv"), ref):
        a, b = getattr(joint, name).cpu() - 0.5, getattr(apart, name).cpu() - 0.5
        assert (a - b).norm() <= 2e-5 * b.norm() + 1e-6 * b.numel() ** 0.5, name
        assert (a - want).norm() <= 1e-2 * want.norm() + 1e-6 * want.numel() ** 0.5, name


def test_joint_backward_under_rope_and_replays(ltr):
    """RoPE's gradient in the dQ blocks, and a captured backward replayed between eager calls."""
    g = torch.Generator().manual_seed(5)
    q, do, k, v = (torch.randn(2, 300, 8, 128, generator=g).to(torch.bfloat16).cuda() for _ in range(4))
    freqs = ltr.precompute_freqs_cis(128, 300)
    table = ltr.rope_table(freqs).cuda()
    assert ltr.attn_plan(2, 8, 8, 128, 300, [300], [0], causal=True, joint=True)["dq"]["kernel"].startswith("bwd_joint")
    def grads(rope):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)]
        x = leaves[0] if rope else ltr.apply_rotary_emb(leaves[0], leaves[0], freqs.cuda())[0]
        ltr.block_attention(x, [leaves[1]], [leaves[2]], [0], causal=True, **(dict(q_rope=table) if rope else {}))[0].backward(do)
        return [t.grad for t in leaves]
    for a, b in zip(grads(True), grads(False)):   # dQ rounded before its rotation, or after
        assert (a.float() - b.float()).norm() <= 5e-3 * b.float().norm()
    with torch.no_grad():
        o, lse = ltr.block_attention(q, [k], [v], [0], causal=True)
    delta, out = torch.empty_like(lse), [torch.empty_like(t) for t in (q, k, v)]
    call = lambda: ltr.attn_bwd_accumulate(q, do, lse, delta, [k], [v], [0], out[0], [out[1]], [out[2]], 0, None, True, o=o, joint=True)
    call()
    want = [t.clone() for t in out]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        for t in out:
            t.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
        call()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
