"""The forward and dQ kernels whose waves share a row group's keys (fwd_bf16_shares_kernel, bwd_dq_shares_kernel): launches with few
query rows, against the dense oracle."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,split,chunks,causal,ks", [
    (128, 2, 16, 16, 700, 0, None, [(700, 0)], True, 2),                              # tails in rows and keys
    (128, 1, 8, 2, 512, 0, None, [(512, 0)], True, 4),
    (128, 1, 4, 4, 33, 100, None, [(31, 0), (97, 31), (64, 90)], True, 2),            # chunks shorter than a tile of all shares
    (128, 1, 4, 2, 200, (40, 1300), 130, [(128, 0), (933, 500), (256, 4000)], True, 4), # two segments, rows that see no key, a chunk no row sees
    (64, 8, 12, 4, 200, 0, None, [(520, 0)], False, 2),
    (64, 1, 8, 1, 100, 0, None, [(300, 50)], True, 4),                                # the first rows see no key
    (64, 1, 4, 2, 65, 0, None, [(65, 0), (1, 65)], False, 4),
])
def test_key_shares_forward_backward(ltr, D, B, Hq, Hkv, Sq, q_pos, split, chunks, causal, ks):
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, [n for n, _ in chunks], [p for _, p in chunks], q_pos, split, causal)
    assert plan["fwd"]["kernel"] == "fwd_bf16_shares_kernel<%d, %d>" % (D, ks) and plan["fwd"]["rows"] == 256 // ks
    assert plan["dq"]["kernel"].startswith("bwd_dq_shares_kernel<%d, " % D)
    g = torch.Generator().manual_seed(D + Sq)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, do = mk(B, Sq, Hq, D), mk(B, Sq, Hq, D)
    total = sum(n for n, _ in chunks)
    k, v = mk(B, total, Hkv, D), mk(B, total, Hkv, D)
    at = [sum(n for n, _ in chunks[:i]) for i in range(len(chunks))]
    cut = lambda t: [t[:, a:a + n] for a, (n, _) in zip(at, chunks)]
    pos = [p for _, p in chunks]
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    rows = torch.arange(Sq)
    qpos = rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    o_ref, lse_ref, dq_ref, _, _ = orc.dense_attention_grads(q.float(), k.float(), v.float(), do.float(), qpos, kpos, causal, dtype=torch.float32)
    qd, kd, vd, dod = q.cuda(), k.cuda(), v.cuda(), do.cuda()
    fin = torch.isfinite(lse_ref)

    def check(o, lse, tol):
        assert (o.cpu().float() - o_ref).abs().max() < tol
        assert torch.equal(torch.isfinite(lse.cpu()), fin) and (lse.cpu()[fin] - lse_ref[fin]).abs().max() < 2e-2

    o, lse = ltr.attn_fwd(qd, cut(kd), cut(vd), pos, q_pos, split, causal)
    check(o, lse, 2e-2)
    # the partial result of one chunk after the other, merged in the epilogue (fp32 O)
    om, lm = ltr.attn_fwd(qd, cut(kd)[:1], cut(vd)[:1], pos[:1], q_pos, split, causal, out_dtype=torch.float32)
    for i in range(1, len(chunks)):
        ltr.attn_fwd(qd, cut(kd)[i:i + 1], cut(vd)[i:i + 1], pos[i:i + 1], q_pos, split, causal, out=om, lse=lm, merge=True)
    check(om, lm, 2e-2)
    # dQ as a bf16 result with DELTA from O, and accumulated in fp32; the two differ by the final rounding only
    delta = torch.empty(lse.shape, dtype=torch.float32, device="cuda")
    dq16 = torch.full(q.shape, 7.0, dtype=torch.bfloat16, device="cuda")
    dq32 = torch.full(q.shape, 0.5, dtype=torch.float32, device="cuda")
    sink = cut(torch.zeros(k.shape, dtype=torch.float32, device="cuda"))
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq16, sink, sink, q_pos, split, causal, do_dkdv=False, o=o)
    assert (delta.cpu() - (do.float() * o.cpu().float()).sum(-1).transpose(1, 2)).abs().max() < 1e-3 * D
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq32, sink, sink, q_pos, split, causal, do_dkdv=False)
    dq32 = dq32.cpu() - 0.5
    assert (dq32 - dq_ref).norm() <= 1e-2 * dq_ref.norm()       # 2.0e-3 .. 3.1e-3: P, dS and the inputs' products in bf16
    # one key lost or taken twice at a border of shares or chunks would hide in that: against the kernels that share nothing.  dQ: the
    # same bf16 P and dS, summed in another order; O: P rounded against another reference (2^-9 of each term, on both sides)
    of, lf = ltr.attn_fwd(qd, cut(kd), cut(vd), pos, q_pos, split, causal, out_dtype=torch.float32)
    o1, l1 = ltr.attn_fwd(qd, cut(kd), cut(vd), pos, q_pos, split, causal, out_dtype=torch.float32, fwd_rows=256)
    assert (of - o1).norm() <= 4e-3 * o1.norm() and (lf.cpu()[fin] - l1.cpu()[fin]).abs().max() <= 2e-4
    dq1 = torch.zeros(q.shape, dtype=torch.float32, device="cuda")
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq1, sink, sink, q_pos, split, causal, do_dkdv=False, dq_rows=256)
    assert (dq32 - dq1.cpu()).norm() <= 1e-5 * dq1.cpu().norm()
    # bf16 rounding (2^-8 of the value) and the cancellation of the accumulator's start value (2^-23 of 0.5 + |dQ|)
    assert ((dq16.cpu().float() - dq32).abs() <= dq32.abs() / 256 + 1e-6).all()


@pytest.mark.parametrize("D,Hq,Hkv,Sq,q_pos,split,chunks", [
    (64, 16, 16, 3900, 0, None, [(3900, 0)]),                                           # an odd number of tiles: the middle one alone
    (128, 16, 16, 3801, 0, None, [(1701, 0), (2100, 1701)]),
    (64, 16, 16, 3840, (0, 5760), 1920, [(1920, 0), (1920, 5760)]),   # a zig-zag share against its own keys
])
def test_key_shares_in_pairs_of_tiles(ltr, D, Hq, Hkv, Sq, q_pos, split, chunks):
    plan = ltr.attn_plan(1, Hq, Hkv, D, Sq, [n for n, _ in chunks], [p for _, p in chunks], q_pos, split, True)
    assert plan["fwd"]["paired"] and plan["dq"]["paired"]
    test_key_shares_forward_backward(ltr, D, 1, Hq, Hkv, Sq, q_pos, split, chunks, True, 2)
