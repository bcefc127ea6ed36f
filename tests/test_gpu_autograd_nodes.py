"""The C++ autograd nodes under what torch may do around them: saved-tensor hooks that hand tensors back in another layout, tables
changed between forward and backward, gradients of gradients of the exchange, empty chunks."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


def _repacked(t):      # a dense copy: slices of one buffer come back with strides of their own
    return t.clone(memory_format=torch.contiguous_format)


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (96, torch.bfloat16), (64, torch.float32)])
def test_saved_tensor_hooks_may_change_strides(ltr, D, dtype):
    g = torch.Generator(device="cuda").manual_seed(D)
    mk = lambda s, h: torch.randn(2, s, h, D, generator=g, device="cuda").to(dtype)
    q0, k0, v0, do = mk(90, 4), mk(170, 2), mk(170, 2), mk(90, 4)
    grads = []
    for hooks in (False, True):
        q, k, v = (t.clone().requires_grad_(True) for t in (q0, k0, v0))
        with torch.autograd.graph.saved_tensors_hooks(_repacked if hooks else (lambda t: t), lambda t: t):
            o, _ = ltr.block_attention(q, [k[:, :70], k[:, 70:]], [v[:, :70], v[:, 70:]], [0, 70], 80, None, True)
        o.backward(do)
        grads.append([q.grad, k.grad, v.grad])
    # the same kernels on the same values: the same bits
    assert all(torch.equal(a, b) for a, b in zip(*grads))


def test_a_rope_table_changed_before_the_backward_is_noticed(ltr):
    q = torch.randn(1, 40, 2, 64, device="cuda", dtype=torch.bfloat16).requires_grad_(True)
    kv = torch.randn(1, 40, 2, 64, device="cuda", dtype=torch.bfloat16)
    table = torch.view_as_real(ltr.precompute_freqs_cis(64, 40, device="cuda")).contiguous()
    o, _ = ltr.block_attention(q, [kv], [kv], [0], causal=True, q_rope=table)
    table.mul_(2)
    with pytest.raises(RuntimeError, match="inplace"):
        o.sum().backward()


def test_exchange_has_second_derivatives_and_keeps_conjugates(ltr):
    grp = ltr.LocalCPGroup(2)
    for f in (ltr._all_to_all, ltr.SeqAllToAll.apply):
        x = torch.randn(2, 1, 6, 4, 8, device="cuda", requires_grad=True)
        gy = torch.randn_like(f(x.detach(), 2, 1, grp)).requires_grad_(True)
        gx, = torch.autograd.grad(f(x, 2, 1, grp), x, gy, create_graph=True)
        c = torch.randn_like(gx)
        gg, = torch.autograd.grad(gx, gy, c)      # the exchange is linear: its transpose's transpose
        assert torch.equal(gg, f(c, 2, 1, grp))
        z = torch.randn(2, 1, 6, 4, 8, device="cuda", dtype=torch.complex64)
        assert torch.equal(f(z.conj(), 2, 1, grp), f(z, 2, 1, grp).conj())


def test_no_query_rows_with_an_empty_chunk(ltr):
    q = torch.randn(1, 0, 2, 64, device="cuda", dtype=torch.bfloat16)
    ks = [torch.randn(1, n, 2, 64, device="cuda", dtype=torch.bfloat16) for n in (0, 5)]
    o, lse = ltr.block_attention(q, ks, ks, [0, 0])
    assert o.shape == (1, 0, 2, 64) and lse.shape == (1, 2, 0)


@pytest.mark.parametrize("D,B,H,Sq,q_pos,chunks,causal,ks", [
    (64, 1, 4, 100, 0, [(100, 0)], True, 4),
    (64, 4, 16, 200, 0, [(150, 0), (50, 150)], True, 2),
    (64, 8, 16, 200, 0, [(33, 0)], False, 1),
    (64, 1, 2, 70, 0, [(64, 40)], True, 4),              # a block of rows that sees no key, and one that sees some
    (128, 8, 16, 131, 5, [(136, 0)], True, 1),
    (128, 1, 4, 65, 0, [(40, 33)], True, 2),
])
def test_fp32_dq_is_stored_and_delta_comes_from_o(ltr, D, B, H, Sq, q_pos, chunks, causal, ks):
    plan = ltr.attn_plan(B, H, H, D, Sq, [n for n, _ in chunks], [p for _, p in chunks], q_pos, None, causal, dtype=torch.float32)
    assert plan["dq"]["kernel"] == "bwd_dq_f32_mfma_kernel<%d, %d>" % (D, ks)
    g = torch.Generator().manual_seed(Sq)
    total, start = sum(n for n, _ in chunks), [sum(n for n, _ in chunks[:i]) for i in range(len(chunks))]
    q, do = (torch.randn(B, Sq, H, D, generator=g) for _ in range(2))
    k, v = (torch.randn(B, total, H, D, generator=g) for _ in range(2))
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    qpos = torch.arange(Sq) + q_pos
    want = orc.dense_attention_grads(q, k, v, do, qpos, kpos, causal, dtype=torch.float64)[2:]
    qd, kd, vd = (t.cuda().requires_grad_(True) for t in (q, k, v))
    poison = [torch.full((1 << 20,), float("nan"), device="cuda") for _ in range(4)]   # freed: the buffers of the call start as NaN
    del poison
    cut = lambda t: [t[:, a:a + n] for a, (n, _) in zip(start, chunks)]
    o, _ = ltr.block_attention(qd, cut(kd), cut(vd), [p for _, p in chunks], q_pos, causal=causal)
    o.backward(do.cuda())
    # fp32 sums of up to 256 terms of order 1
    for got, ref in zip((qd.grad, kd.grad, vd.grad), want):
        assert (got.cpu().double() - ref).norm() <= 5e-6 * ref.norm() and torch.isfinite(got).all()
    unseen = (qpos < kpos.min()) if causal else torch.zeros(Sq, dtype=torch.bool)
    assert not qd.grad.cpu()[:, unseen].any()
