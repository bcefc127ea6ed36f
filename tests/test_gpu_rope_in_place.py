"""q rotated in place by the forward kernel's prologue (q_rot == q), at sizes whose launches would otherwise share keys: several waves of
a block read a row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,B,Hq,Hkv,Sq", [(128, 1, 8, 2, 512), (128, 2, 16, 16, 700), (64, 1, 8, 1, 100), (64, 8, 12, 4, 200)])
def test_rotation_in_place_matches_the_copy(ltr, D, B, Hq, Hkv, Sq):
    plan = ltr.attn_plan(B, Hq, Hkv, D, Sq, [Sq], [0], causal=True)
    assert "shares" in plan["fwd"]["kernel"]
    g = torch.Generator(device="cuda").manual_seed(D)
    q, k, v = (torch.randn(B, Sq, h, D, device="cuda", generator=g).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    table = ltr.rope_table(ltr.precompute_freqs_cis(D, Sq, device="cuda"))
    rot = torch.empty_like(q)
    o, lse = ltr.attn_fwd(q, [k], [v], [0], causal=True, q_rope=table, q_rot_out=rot, fwd_rows=256)
    inplace = q.clone()
    o2, lse2 = ltr.attn_fwd(inplace, [k], [v], [0], causal=True, q_rope=table, q_rot_out=inplace)
    assert torch.equal(inplace, rot) and torch.equal(o, o2) and torch.equal(lse, lse2)
