"""Head dims other than 64 / 128 in the kernels themselves (LTR_HEAD_COLS: columns past the head dim cleared on chip), against the
dense oracle and against the zero-padded path."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double().cpu() - b.double()).norm() / b.double().norm()).item()


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,lens,causal,rope", [
    (8, 1, 2, 1, 70, 0, [70], True, False),              # one 16-byte chunk per row
    (56, 2, 4, 2, 130, 40, [33, 137], True, True),
    (72, 2, 4, 4, 300, 0, [300], False, False),          # one chunk past 64
    (120, 1, 8, 2, 515, 0, [300, 215], True, True),      # one chunk short of 128
    (96, 16, 32, 32, 520, 0, [520], True, False),        # 256-row blocks, tiles paired
    (40, 16, 32, 8, 300, 0, [300], True, False),
])
def test_head_cols_forward_backward(ltr, D, B, Hq, Hkv, Sq, q_pos, lens, causal, rope):
    g = torch.Generator().manual_seed(D)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, do = mk(B, Sq, Hq, D), mk(B, Sq, Hq, D)
    k, v = mk(B, sum(lens), Hkv, D), mk(B, sum(lens), Hkv, D)
    at = [sum(lens[:i]) for i in range(len(lens))]
    cut = lambda t: [t[:, a:a + n] for a, n in zip(at, lens)]
    fc = orc.precompute_freqs_cis(D, q_pos + Sq)
    table = ltr.rope_table(fc.cuda()) if rope else None
    from lightron_amd import attention as A
    res = []
    for native in (True, False):
        qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
        assert A._native_cols(qd, cut(kd), cut(vd), None)
        A.USE_CPP_NODE = native
        try:
            import warnings
            with warnings.catch_warnings():
                warnings.simplefilter("ignore")
                o, lse = ltr.block_attention(qd, cut(kd), cut(vd), at, q_pos, None, causal, q_rope=table)
            assert ("Chunk" in o.grad_fn.name()) == native
            o.backward(do.cuda())
        finally:
            A.USE_CPP_NODE = True
        res.append((o.detach(), lse, qd.grad, kd.grad, vd.grad))
    # the same arithmetic on the same columns; the shares a launch takes may differ between the two, the rounding then too
    for x, y in zip(*res):
        assert _rel(x, y.cpu()) < 4e-3
    rows = slice(0, 2)                                    # the oracle on the first batch entries
    qr = q[rows].float()
    if rope:
        qr = orc.apply_rotary_emb(q[rows], q[rows], fc[q_pos:q_pos + Sq])[0].float()
    qr.requires_grad_(True)
    ref = orc.dense_attention_grads(qr, k[rows].float(), v[rows].float(), do[rows].float(), torch.arange(Sq) + q_pos, torch.arange(sum(lens)), causal,
                                    dtype=torch.float32)
    o, lse, dq, dk, dv = (t[rows].cpu() for t in res[0])
    assert (o.float() - ref[0].detach()).abs().max() < 2e-2 and (lse - ref[1].detach()).abs().max() < 2e-2
    if not rope:                                          # the oracle's dQ is that of the rotated q
        assert _rel(dq, ref[2].detach()) < 5e-2
    assert _rel(dk, ref[3].detach()) < 5e-2 and _rel(dv, ref[4].detach()) < 5e-2


def test_head_cols_leave_neighbours_alone(ltr):
    """Heads packed side by side in one row: nothing is read into, or written past, a head's own columns."""
    B, S, H, D = 2, 140, 3, 72
    g = torch.Generator().manual_seed(4)
    qkv = torch.randn(B, S, 3, H, D, generator=g).to(torch.bfloat16).cuda()
    q, k, v = (qkv[:, :, i].requires_grad_(True) for i in range(3))
    big = torch.full((B, S, H, 128), 3.0, dtype=torch.bfloat16, device="cuda")
    q.retain_grad(), k.retain_grad(), v.retain_grad()
    o, _ = ltr.block_attention(q, [k], [v], [0], causal=True)
    o.backward(torch.ones_like(o))
    qc, kc, vc = (t.detach().contiguous().requires_grad_(True) for t in (q, k, v))
    oc, _ = ltr.block_attention(qc, [kc], [vc], [0], causal=True)
    oc.backward(torch.ones_like(oc))
    assert torch.equal(o, oc) and torch.equal(q.grad, qc.grad) and torch.equal(k.grad, kc.grad) and torch.equal(v.grad, vc.grad)
    # an output whose rows are wider than the head: the low-level call writes D columns of each row and no more
    from lightron_amd import _lib as L
    import ctypes
    a = L.FwdArgs()
    lse = torch.empty(B, H, S, device="cuda")
    a.q, a.o, a.lse = qc.data_ptr(), big.data_ptr(), lse.data_ptr()
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.q_split, a.n_chunks = B, H, H, D, S, S, 1
    for name, t in (("q_stride", qc), ("o_stride", big), ("k_stride", kc), ("v_stride", vc)):
        for i in range(3):
            getattr(a, name)[i] = t.stride(i)
    a.scale, a.io_dtype, a.o_dtype, a.flags = D ** -0.5, L.LTR_BF16, L.LTR_BF16, L.LTR_CAUSAL | L.LTR_HEAD_COLS
    a.chunk[0].k, a.chunk[0].v, a.chunk[0].sk = kc.data_ptr(), vc.data_ptr(), S
    L.check(L.load().ltr_attn_fwd(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "ltr_attn_fwd")
    torch.cuda.synchronize()
    assert torch.equal(big[..., :D], oc.detach()) and (big[..., D:] == 3.0).all()
