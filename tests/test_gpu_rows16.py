"""fwd_f32_mfma_kernel<64, 4> / bwd_dq_f32_mfma_kernel<64, 4> (groups of 16 rows, the keys of a step shared by four waves of 32),
which fp32 launches of the fewest rows take: against the dense oracle in 64 bits at the edges of their tiles."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,Sq,q_pos,split,chunks,causal", [
    (1, 1, 1, 1, 0, None, [(1, 0)], True),
    (1, 2, 2, 15, 0, None, [(15, 0)], True),
    (2, 4, 2, 16, 16, None, [(16, 0), (16, 16)], True),
    (1, 3, 1, 17, 100, None, [(31, 0), (33, 90), (1, 300)], True),                # part of a wave's keys, a chunk that no row sees
    (2, 4, 4, 100, (40, 300), 33, [(127, 0), (129, 100), (64, 280)], True),       # two segments in one group, a key past a step
    (1, 8, 4, 47, 0, None, [(65, 0), (128, 65), (97, 193)], False),               # waves past the end of a chunk
    (2, 8, 8, 256, 0, None, [(256, 0)], True),                                    # as many blocks as CUs
    (1, 2, 2, 40, 0, None, [(300, 20)], True),                                    # groups of rows that see no key
])
def test_rows16(ltr, B, Hq, Hkv, Sq, q_pos, split, chunks, causal):
    D, pos, lens = 64, [p for _, p in chunks], [n for n, _ in chunks]
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, lens, pos, q_pos, split, causal, dtype=torch.float32)
    assert plan["fwd"]["kernel"] == "fwd_f32_mfma_kernel<64, 4>" and plan["dq"]["kernel"] == "bwd_dq_f32_mfma_kernel<64, 4>"
    assert plan["fwd"]["rows"] == 16 and plan["dq"]["rows"] == 16 and plan["fwd"]["blocks"] == B * Hq * ((Sq + 15) // 16)
    total, at = sum(lens), [sum(lens[:i]) for i in range(len(lens))]
    g = torch.Generator().manual_seed(Sq)
    mk = lambda s, h: torch.randn(B, s, h, D, generator=g)
    q, do, k, v = mk(Sq, Hq), mk(Sq, Hq), mk(total, Hkv), mk(total, Hkv)
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    rows = torch.arange(Sq)
    qpos = rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    o_ref, lse_ref, *grads = orc.dense_attention_grads(q, k, v, do, qpos, kpos, causal, dtype=torch.float64)
    cut = lambda t: [t[:, a:a + n] for a, n in zip(at, lens)]
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o, lse = ltr.block_attention(qd, cut(kd), cut(vd), pos, q_pos, split, causal=causal)
    om, lm = ltr.attn_fwd(qd.detach(), cut(kd.detach())[:1], cut(vd.detach())[:1], pos[:1], q_pos, split, causal)
    for i in range(1, len(chunks)):   # one chunk after the other, merged in the epilogue
        ltr.attn_fwd(qd.detach(), cut(kd.detach())[i:i + 1], cut(vd.detach())[i:i + 1], pos[i:i + 1], q_pos, split, causal, out=om, lse=lm, merge=True)
    fin = torch.isfinite(lse_ref)
    for oo, ll in ((o.detach(), lse.detach()), (om, lm)):
        # fp32 sums of up to 384 terms: some 2^-24 sqrt(384) = 1.2e-6 of the largest score (about 5) and of the outputs
        assert (oo.cpu().double() - o_ref).abs().max() < 1e-5
        assert torch.equal(torch.isfinite(ll.cpu()), fin) and (ll.cpu().double()[fin] - lse_ref[fin]).abs().max() < 1e-5
    o.backward(do.cuda())
    # dS = P (dO . v - DELTA): a row that sees one key has a gradient of zero, the difference of two fp32 sums of 64 products (about 8, rounded
    # to some 2^-24 of it: 1e-6 of a unit), times the scale and a key of norm 8: 1e-6 per row, and the rows' dO are of norm 8 (5e-6 / 8 of it)
    near = do.double().norm() / 8
    for got, ref in zip((qd.grad, kd.grad, vd.grad), grads):
        assert (got.cpu().double() - ref).norm() <= 5e-6 * (ref.norm() + near) and torch.isfinite(got).all()
    # dQ into an accumulator with values in it, DELTA from its own kernel
    acc = torch.ones(B, Sq, Hq, D, device="cuda")
    dk, dv = torch.zeros_like(kd), torch.zeros_like(vd)
    od = o.detach()
    ltr.attn_bwd_accumulate(qd.detach(), do.cuda(), lse.detach(), ltr.attn_delta(od, do.cuda()), cut(kd.detach()), cut(vd.detach()), pos, acc, cut(dk), cut(dv),
                            q_pos, split, causal)
    assert (acc.cpu().double() - 1 - grads[0]).norm() <= 5e-6 * ((1 + grads[0]).norm() + near)


@pytest.mark.parametrize("D,pairs,Sq,rows", [
    (64, 16, 256, 16), (64, 16, 257, 32), (64, 17, 240, 16), (64, 255, 16, 16), (64, 256, 16, 128), (64, 1, 4096, 16), (64, 1, 4097, 32),
    (64, 8, 1024, 32), (64, 255, 17, 32), (128, 1, 1, 64),
])
def test_rows16_where_one_round_of_256_blocks_holds_the_launch(ltr, D, pairs, Sq, rows):
    plan = ltr.attn_plan(1, pairs, pairs, D, Sq, [64], [0], 0, None, True, dtype=torch.float32)
    if plan["compute_units"] == 256:
        assert plan["fwd"]["rows"] == rows and plan["dq"]["rows"] == rows
