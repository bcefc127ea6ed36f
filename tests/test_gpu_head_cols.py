"""Head dims other than 64 / 128 in the kernels themselves (LTR_HEAD_COLS: columns past the head dim cleared on chip), against the
dense oracle and against the zero-padded path."""
import pytest
import torch

from attn_abi import backward
from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double().cpu() - b.double()).norm() / b.double().norm()).item()


def _kernels(ltr, D, B, Hq, Hkv, Sq, q_pos, lens, causal):
    """(key shares of the forward, of dQ, blocks per key tile of dK/dV, tiles in pairs) of the padded kernels this problem runs in where its
    backward is two launches, and the kernel that block_attention's backward takes for both, if it does."""
    at = [sum(lens[:i]) for i in range(len(lens))]
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, lens, at, q_pos, None, causal, share_keys=True)
    width = 64 if D < 64 else 128
    assert plan["dkdv"]["kernel"] == "bwd_dkdv_pad_kernel<%d>" % width
    shares = [256 // plan[x]["rows"] for x in ("fwd", "dq")]
    assert [plan[x]["kernel"] for x in ("fwd", "dq")] == ["%s_pad_kernel<%d, %d>" % (n, width, ks) for n, ks in zip(("fwd_bf16", "bwd_dq"), shares)]
    assert plan["fwd"]["paired"] == plan["dq"]["paired"]
    both = ltr.attn_plan(B, Hq, Hkv, D, Sq, lens, at, q_pos, None, causal, share_keys=True, joint=True)
    joint = both["dq"]["kernel"] if both["dq"]["kernel"] == both["dkdv"]["kernel"] else ""
    assert joint or (both["dq"], both["dkdv"]) == (plan["dq"], plan["dkdv"])
    return (*shares, plan["dkdv"]["blocks_per_tile"], plan["fwd"]["paired"]), joint


def _launches_apart(plan, width, ks, blocks_per_tile, paired):
    """A backward ran dQ and dK/dV in the two padded kernels, with these shares."""
    assert (plan.dq, plan.dkdv) == ("bwd_dq_pad_kernel<%d, %d>" % (width, ks), "bwd_dkdv_pad_kernel<%d>" % width)
    assert (plan.rows, plan.blocks_per_tile, plan.paired) == (256 // ks, blocks_per_tile, paired)


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,q_pos,lens,causal,rope,kernels,joint", [
    (8, 1, 2, 1, 70, 0, [70], True, False, (4, 4, 4, False), "bwd_joint_delta_pad_kernel<64>"),              # one 16-byte chunk per row
    (56, 2, 4, 2, 130, 40, [33, 137], True, True, (4, 4, 4, False), "bwd_joint_delta_pad_kernel<64>"),
    (72, 2, 4, 4, 300, 0, [300], False, False, (2, 4, 1, False), "bwd_joint_pad_kernel<128, 2>"),          # one chunk past 64
    (120, 1, 8, 2, 515, 0, [300, 215], True, True, (4, 4, 16, False), "bwd_joint_pad_kernel<128, 2>"),     # one chunk short of 128
    (96, 16, 32, 32, 520, 0, [520], True, False, (1, 1, 1, True), ""),         # 256-row blocks, tiles paired
    (40, 16, 32, 8, 300, 0, [300], True, False, (1, 1, 1, False), ""),
    (80, 2, 16, 16, 600, 0, [600], True, True, (2, 2, 1, False), "bwd_joint_pad_kernel<128, 2>"),
    (32, 8, 12, 4, 200, 0, [200], False, False, (2, 2, 2, False), "bwd_joint_pad_kernel<64, 1>"),
])
def test_head_cols_forward_backward(ltr, D, B, Hq, Hkv, Sq, q_pos, lens, causal, rope, kernels, joint):
    """block_attention in the kernels that it takes, and the backward of the same problem in two launches."""
    assert _kernels(ltr, D, B, Hq, Hkv, Sq, q_pos, lens, causal) == (kernels, joint)
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
        assert _rel(dq, ref[2].detach()) < 1e-2
    assert _rel(dk, ref[3].detach()) < 1e-2 and _rel(dv, ref[4].detach()) < 1e-2
    qr = ltr.apply_rotary_emb(q.cuda(), q.cuda(), fc[q_pos:q_pos + Sq].cuda())[0] if rope else q.cuda()
    two = backward(qr, do.cuda(), res[0][0], res[0][1], cut(k.cuda()), cut(v.cuda()), at, q_pos, None, causal, fill=7.0)
    _launches_apart(two.plan, 64 if D < 64 else 128, *kernels[1:])
    for got, want in zip((two.dq, two.dk, two.dv), ref[2:]):
        assert _rel(got[rows], want.detach()) < 1e-2


@pytest.mark.parametrize("D,Sq,lens,joint", [(96, 3801, [1701, 2100], "bwd_joint_pad_kernel<128, 1>"), (104, 3801, [1701, 2100], "bwd_joint_pad_kernel<128, 1>"),
                                             (56, 3900, [3900], ""), (64, 3900, [3900], "")])
def test_head_cols_in_pairs_of_tiles(ltr, D, Sq, lens, joint):
    """Two key shares and a late and an early q tile per block: the columns past the head dim are cleared again between the two.
    (D = 64: the check of this test's own reference, the kernels without padding.)"""
    H = 16
    if D != 64:
        assert _kernels(ltr, D, 1, H, H, Sq, 0, lens, True) == ((2, 2, 1, True), joint)
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v, do = (torch.randn(1, Sq, H, D, device="cuda", generator=g).to(torch.bfloat16) for _ in range(4))
    at = [sum(lens[:i]) for i in range(len(lens))]
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    o, lse = ltr.block_attention(q, [k[:, a:a + n] for a, n in zip(at, lens)], [v[:, a:a + n] for a, n in zip(at, lens)], at, causal=True)
    o.backward(do)
    h = slice(0, 2)                                       # the oracle on two heads
    ref = orc.dense_attention_grads(*(t.detach()[:, :, h].float().cpu() for t in (q, k, v, do)), torch.arange(Sq), torch.arange(Sq), True, dtype=torch.float32)
    # scores carry the rounding of q times the scale to bf16: 2^-9 of |q||k| scale, 1.1e-3 rms, 5e-3 at the worst of the rows with one key
    assert (lse[:, h].cpu() - ref[1]).abs().max() < 1e-2
    assert _rel(o.detach()[:, :, h], ref[0]) < 1e-2
    for t, r in zip(leaves, ref[2:]):
        assert _rel(t.grad[:, :, h], r) < 1e-2
    # and every head against the kernels that share no keys and pair no tiles: zero columns up to the next width, 256-row blocks
    W = 64 if D <= 64 else 128
    pad = lambda t: torch.nn.functional.pad(t.detach(), (0, W - D))
    cut = lambda t: [t[:, a:a + n] for a, n in zip(at, lens)]
    qp, kp, vp, dop = (pad(t) for t in (q, k, v, do))
    o1, l1 = ltr.attn_fwd(qp, cut(kp), cut(vp), at, causal=True, scale=D ** -0.5, fwd_rows=256)
    assert _rel(o.detach(), o1[..., :D].cpu()) < 4e-3 and (lse - l1).abs().max() < 2e-4
    dq1 = torch.zeros(qp.shape, dtype=torch.float32, device="cuda")
    sink = cut(torch.zeros(kp.shape, dtype=torch.float32, device="cuda"))
    ltr.attn_bwd_accumulate(qp, dop, l1, ltr.attn_delta(o1, dop), cut(kp), cut(vp), at, dq1, sink, sink, causal=True, scale=D ** -0.5, do_dkdv=False, dq_rows=256)
    assert _rel(q.grad, dq1[..., :D].cpu()) < 4e-3        # the bf16 rounding of the result (2^-9) and of O behind DELTA
    if D == 64:
        return
    two = backward(q.detach(), do, o.detach(), lse, cut(k.detach()), cut(v.detach()), at, causal=True, fill=7.0)
    _launches_apart(two.plan, W, 2, 1, True)
    assert _rel(two.dq, dq1[..., :D].cpu()) < 4e-3
    # the same sums in another order: a bf16 result one step away (2^-8 of it at most) in fewer than one of sixteen
    for got, want, r in zip((two.dq, two.dk, two.dv), (q.grad, k.grad, v.grad), ref[2:]):
        assert _rel(got[:, :, h], r) < 1e-2 and _rel(got, want.cpu()) < 1e-3


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq,causal,kernels", [
    (96, 1, 8, 2, 515, True, (4, 16, False)), (112, 1, 8, 2, 515, True, (4, 16, False)),
    (88, 2, 16, 16, 600, True, (2, 1, False)), (104, 2, 16, 16, 600, True, (2, 1, False)),
    (72, 1, 16, 4, 260, False, (4, 8, False)), (120, 1, 16, 4, 260, False, (4, 8, False)),
])
def test_backward_in_two_launches_on_both_sides_of_column_96(ltr, D, B, Hq, Hkv, Sq, causal, kernels):
    """Two and four key shares of dQ and shared key tiles of dK/dV, in three and in four blocks of columns."""
    g = torch.Generator().manual_seed(D)
    q, do = (torch.randn(B, Sq, Hq, D, generator=g).to(torch.bfloat16) for _ in range(2))
    k, v = (torch.randn(B, Sq, Hkv, D, generator=g).to(torch.bfloat16) for _ in range(2))
    pos = torch.arange(Sq)
    ref = orc.dense_attention_grads(q.float(), k.float(), v.float(), do.float(), pos, pos, causal, dtype=torch.float32)
    o, lse = (t.detach() for t in ltr.block_attention(q.cuda(), [k.cuda()], [v.cuda()], [0], causal=causal))
    two = backward(q.cuda(), do.cuda(), o, lse, [k.cuda()], [v.cuda()], [0], causal=causal, fill=7.0)
    _launches_apart(two.plan, 128, *kernels)
    for got, want in zip((two.dq, two.dk, two.dv), ref[2:]):
        assert _rel(got, want) < 1e-2
        for c in range(0, D, 8):
            assert _rel(got[..., c:c + 8], want[..., c:c + 8]) < 2e-2, c


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
