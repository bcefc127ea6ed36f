"""DELTA = rowsum(dO * O) in fp32: no sum of more than D / 16 terms in a row, wherever it is computed."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _summed_in(o, do, chains):
    """rms error against fp64 of a row sum made of `chains` serial fp32 sums, added up as a tree."""
    terms = (o.double() * do.double()).float().unflatten(-1, (chains, -1))      # the rounding of the products is an fma's at most
    acc = terms[..., 0]
    for i in range(1, terms.shape[-1]):
        acc = acc + terms[..., i]
    while acc.shape[-1] > 1:
        acc = acc[..., ::2] + acc[..., 1::2]
    return (acc[..., 0].double() - (o.double() * do.double()).sum(-1)).pow(2).mean().sqrt().item()


@pytest.mark.parametrize("D", [64, 128])
def test_delta_error_is_that_of_sixteen_sums(ltr, D):
    from lightron_amd import _lib as L
    B, S, H = 2, 700, 6
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v, do = (torch.randn(B, S, H, D, device="cuda", generator=g) for _ in range(4))
    o, lse = ltr.attn_fwd(q, [k], [v], [0])
    o = torch.randn(o.shape, device="cuda", generator=g)      # O of unit size: DELTA's own rounding, not the softmax's
    want = (o.double() * do.double()).sum(-1).transpose(1, 2)
    bound = 1.15 * _summed_in(o, do, 16)        # 8400 rows: the rms of two such errors differs by 2 %; serial halves are 1.5 - 1.9 times off
    rms = lambda d: (d.double() - want).pow(2).mean().sqrt().item()
    assert rms(ltr.attn_delta(o, do)) <= bound
    # left by the dQ kernel (LTR_DQ_F32_RESULT)
    delta, dq = torch.full(lse.shape, 9.0, device="cuda"), torch.empty_like(q)
    a = L.BwdArgs()
    a.q, a.d_o, a.lse, a.delta, a.dq, a.o = (t.data_ptr() for t in (q, do, lse, delta, dq, o))
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.q_split, a.n_chunks, a.io_dtype = B, H, H, D, S, S, 1, L.LTR_F32
    for name in ("q_stride", "do_stride", "dq_stride", "k_stride", "v_stride", "dk_stride", "dv_stride", "o_stride"):
        for i in range(3):
            getattr(a, name)[i] = q.stride(i)
    a.scale, a.flags = D ** -0.5, L.LTR_DQ_F32_RESULT | L.LTR_NO_DKDV
    a.chunk[0].k, a.chunk[0].v, a.chunk[0].sk = k.data_ptr(), v.data_ptr(), S
    L.check(L.load().ltr_attn_bwd(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "ltr_attn_bwd")
    assert rms(delta) <= bound


@pytest.mark.parametrize("D", [8, 40, 64, 72, 128])
@pytest.mark.parametrize("B,S,H", [(1, 1, 1), (2, 31, 1), (1, 33, 3), (3, 65, 5)])   # rows on both sides of a block's 32 or 64
def test_delta_of_aligned_bf16_is_that_of_the_general_kernel(ltr, D, B, S, H):
    g = torch.Generator(device="cuda").manual_seed(D + S)
    wide = torch.randn(2, B, S, H + 1, D, device="cuda", generator=g).to(torch.bfloat16)
    o, do = wide[0, :, :, 1:], wide[1, :, :, :H]              # strides of their own
    shifted = torch.empty(o.numel() + 1, device="cuda", dtype=torch.bfloat16)[1:].view(o.shape)   # 2 bytes off: the general kernel
    shifted.copy_(o)
    got = ltr.attn_delta(o, do)
    assert torch.equal(got, ltr.attn_delta(shifted, do))
    want = (o.double() * do.double()).sum(-1).transpose(1, 2)
    bound = D * 2.0 ** -24 * (o.double() * do.double()).abs().sum(-1).transpose(1, 2)   # D roundings of fp32, each of at most the sum of sizes
    assert ((got.double() - want).abs() <= bound).all()
