"""Head dims above 64 in the kernels of width 128: three blocks of 32 columns up to 96, four above.  Forward and backward against the dense
oracle on both sides of the edge, whole launches and shared ones."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [72, 88, 96, 104])
@pytest.mark.parametrize("B,Hq,Hkv,S,causal,kernels", [
    (1, 8, 2, 193, True, ("fwd_bf16_pad_kernel<128, 2>", "bwd_joint_pad_kernel<128, 2>", "bwd_joint_pad_kernel<128, 2>", 8)),
    (2, 8, 8, 260, False, ("fwd_bf16_pad_kernel<128, 2>", "bwd_joint_pad_kernel<128, 2>", "bwd_joint_pad_kernel<128, 2>", 1)),
    (8, 32, 8, 300, True, ("fwd_bf16_pad_kernel<128, 1>", "bwd_dq_pad_kernel<128, 1>", "bwd_dkdv_pad_kernel<128>", 1)),
])
def test_columns(ltr, D, B, Hq, Hkv, S, causal, kernels):
    plan = ltr.attn_plan(B, Hq, Hkv, D, S, [S], [0], causal=causal, share_keys=True, joint=True)
    assert (plan["fwd"]["kernel"], plan["dq"]["kernel"], plan["dkdv"]["kernel"], plan["dkdv"]["blocks_per_tile"]) == kernels
    g = torch.Generator().manual_seed(D)
    mk = lambda h: torch.randn(B, S, h, D, generator=g).to(torch.bfloat16)
    q, k, v, do = mk(Hq), mk(Hkv), mk(Hkv), mk(Hq)
    pos = torch.arange(S)
    o_ref, lse_ref, *ref = orc.dense_attention_grads(q.float(), k.float(), v.float(), do.float(), pos, pos, causal, dtype=torch.float32)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    o, lse = ltr.block_attention(leaves[0], [leaves[1]], [leaves[2]], [0], causal=causal)
    o.backward(do.cuda())
    assert (lse.detach().cpu() - lse_ref).abs().max() < 4.1e-3   # the sum of a row is that of P rounded to bf16: 2^-8 of one key's
    # bf16 operands, P and results: 2e-3 .. 3.1e-3 of the norm, of every block of 8 columns as well
    for name, got, want in zip(("o", "dq", "dk", "dv"), (o.detach(), *(t.grad for t in leaves)), (o_ref, *ref)):
        got = got.cpu().float()
        assert (got - want).norm() <= 1e-2 * want.norm(), name
        for c in range(0, D, 8):
            assert (got[..., c:c + 8] - want[..., c:c + 8]).norm() <= 2e-2 * want[..., c:c + 8].norm(), (name, c)
