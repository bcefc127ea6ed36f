"""fwd_bf16_w4_kernel / bwd_dq_w4_kernel (blocks of four waves and 128 rows, several per CU), which launches of many short blocks take:
against the dense oracle at the edges of their tiles (128 rows per block, 32 per wave, 64 keys)."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,split,chunks,causal", [
    (64, 40, 16, 16, 140, 0, None, [(140, 0)], True),                               # a second tile of 12 rows
    (64, 37, 12, 12, 257, 0, None, [(257, 0)], True),                               # one row and key past two tiles; 444 pairs, not a multiple of 8
    (64, 24, 24, 12, 150, (40, 300), 33, [(31, 0), (130, 31), (64, 500)], True),    # two segments, chunk tails, keys no row sees, rows that see few
    (64, 20, 32, 8, 129, 0, None, [(65, 0), (64, 65)], False),                      # no mask, one row past a tile
    (128, 24, 16, 16, 300, 0, None, [(300, 0)], True),
    (128, 19, 24, 12, 290, 7, None, [(297, 0)], True),                              # q positions past the keys' start, two q heads per kv head
])
def test_four_waves(ltr, D, B, Hq, Hkv, Sq, q_pos, split, chunks, causal):
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, [n for n, _ in chunks], [p for _, p in chunks], q_pos, split, causal)
    assert plan["fwd"]["kernel"] == "fwd_bf16_w4_kernel<%d>" % D and plan["fwd"]["rows"] == 128
    assert plan["dq"]["kernel"] == "bwd_dq_w4_kernel<%d>" % D and plan["dq"]["rows"] == 128
    total = sum(n for n, _ in chunks)
    g = torch.Generator().manual_seed(Sq)
    mk = lambda s, h: torch.randn(B, s, h, D, generator=g).to(torch.bfloat16)
    q, do, k, v = mk(Sq, Hq), mk(Sq, Hq), mk(total, Hkv), mk(total, Hkv)
    at = [sum(n for n, _ in chunks[:i]) for i in range(len(chunks))]
    cut = lambda t: [t[:, a:a + n] for a, (n, _) in zip(at, chunks)]
    pos = [p for _, p in chunks]
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    rows = torch.arange(Sq)
    qpos = rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    o_ref, lse_ref, dq_ref, _, _ = orc.dense_attention_grads(q.float(), k.float(), v.float(), do.float(), qpos, kpos, causal, dtype=torch.float32)
    qd, kd, vd, dod = q.cuda(), k.cuda(), v.cuda(), do.cuda()
    o, lse = ltr.attn_fwd(qd, cut(kd), cut(vd), pos, q_pos, split, causal)
    assert (o.cpu().float() - o_ref).abs().max() < 2e-2 and (lse.cpu() - lse_ref).abs().max() < 2e-2
    # one chunk after the other, merged in the epilogue (fp32 O)
    om, lm = ltr.attn_fwd(qd, cut(kd)[:1], cut(vd)[:1], pos[:1], q_pos, split, causal, out_dtype=torch.float32)
    for i in range(1, len(chunks)):
        ltr.attn_fwd(qd, cut(kd)[i:i + 1], cut(vd)[i:i + 1], pos[i:i + 1], q_pos, split, causal, out=om, lse=lm, merge=True)
    assert (om.cpu() - o_ref).abs().max() < 2e-2 and (lm.cpu() - lse_ref).abs().max() < 2e-2
    delta = torch.empty(lse.shape, dtype=torch.float32, device="cuda")
    dq16 = torch.full(q.shape, 7.0, dtype=torch.bfloat16, device="cuda")
    dq32 = torch.full(q.shape, 0.5, dtype=torch.float32, device="cuda")
    sink = cut(torch.zeros(k.shape, dtype=torch.float32, device="cuda"))
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq16, sink, sink, q_pos, split, causal, do_dkdv=False, o=o)
    assert (delta.cpu() - (do.float() * o.cpu().float()).sum(-1).transpose(1, 2)).abs().max() < 1e-3 * D
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq32, sink, sink, q_pos, split, causal, do_dkdv=False)
    dq32 = dq32.cpu() - 0.5
    # bf16 P, dS and products: 2e-3 .. 3.1e-3 of the norm, of every group of 32 rows (a wave's) as well
    assert (dq32 - dq_ref).norm() <= 1e-2 * dq_ref.norm()
    for first in range(0, Sq, 32):
        a, b = dq32[:, first:first + 32], dq_ref[:, first:first + 32]
        assert (a - b).norm() <= 3e-2 * b.norm() + 1e-5, first
    # against the eight-wave blocks: the same bf16 P and dS, summed in another order
    dq1 = torch.zeros(q.shape, dtype=torch.float32, device="cuda")
    ltr.attn_bwd_accumulate(qd, dod, lse, delta, cut(kd), cut(vd), pos, dq1, sink, sink, q_pos, split, causal, do_dkdv=False, dq_rows=256)
    assert (dq32 - dq1.cpu()).norm() <= 1e-5 * dq1.cpu().norm()
    # bf16 rounding (2^-8 of the value) and the cancellation of the accumulator's start value (2^-23 of 0.5 + |dQ|)
    assert ((dq16.cpu().float() - dq32).abs() <= dq32.abs() / 256 + 1e-6).all()


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,split", [
    (64, 40, 16, 16, 140, 0, None),
    (64, 24, 24, 12, 150, (40, 300), 33),        # two segments: a wave's rows from both
    (128, 24, 16, 16, 300, 0, None),
    (128, 19, 24, 12, 290, 7, None),
])
def test_four_waves_with_rope(ltr, D, B, Hq, Hkv, Sq, q_pos, split):
    """q rotated in the prologue (into a copy and in place) and dQ rotated back in the epilogue, against launches of the same kernels on q rotated
    beforehand."""
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    total = max(qp) + Sq
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, [total], [0], q_pos, split, True)
    assert plan["fwd"]["kernel"] == "fwd_bf16_w4_kernel<%d>" % D and plan["dq"]["kernel"] == "bwd_dq_w4_kernel<%d>" % D
    g = torch.Generator(device="cuda").manual_seed(Sq)
    q, do, k, v = (torch.randn(B, s, h, D, generator=g, device="cuda").to(torch.bfloat16) for s, h in ((Sq, Hq), (Sq, Hq), (total, Hkv), (total, Hkv)))
    freqs = orc.precompute_freqs_cis(D, total)
    rows = torch.arange(Sq)
    at = freqs[rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])]
    q_in = orc.apply_rotary_emb(q.cpu(), q.cpu(), at)[0].cuda()
    table = ltr.rope_table(freqs.cuda())
    o_ref, lse_ref = ltr.attn_fwd(q_in, [k], [v], [0], q_pos, split, True)
    rot, inplace = torch.full_like(q, float("nan")), q.clone()
    for src, dst in ((q, rot), (inplace, inplace), (q, None)):
        o, lse = ltr.attn_fwd(src, [k], [v], [0], q_pos, split, True, q_rope=table, q_rot_out=dst)
        assert torch.equal(o, o_ref) and torch.equal(lse, lse_ref)
        assert dst is None or torch.equal(dst, q_in)
    delta = torch.empty(lse.shape, dtype=torch.float32, device="cuda")
    sink = torch.zeros(k.shape, dtype=torch.float32, device="cuda")
    plain, turned = (torch.full(q.shape, start, dtype=torch.float32, device="cuda") for start in (0.0, 0.5))
    turned16 = torch.empty_like(q)
    for dq, kw in ((plain, {}), (turned, dict(dq_rope=table)), (turned16, dict(dq_rope=table))):
        ltr.attn_bwd_accumulate(rot, do, lse, delta, [k], [v], [0], dq, [sink], [sink], q_pos, split, True, do_dkdv=False, o=o, **kw)
    want = orc.apply_rotary_emb(plain.cpu(), plain.cpu(), at.conj())[0]
    got = turned.cpu() - 0.5
    # four fp32 products per pair of columns, and the cancellation of the accumulator's start value (2^-23 of 0.5 + |dQ|)
    assert ((got - want).abs() <= 2e-6 * (0.5 + want.abs())).all()
    assert ((turned16.cpu().float() - want).abs() <= want.abs() / 256 + 2e-6).all()
