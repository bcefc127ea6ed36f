"""Key tiles of the dK/dV kernels shared by several blocks (ltr_attn_bwd_ws): partial sums in a workspace and the reduction
kernel, against the unshared launch and the dense oracle."""
import ctypes

import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


def _randn(shape, g, dtype):
    return torch.randn(shape, generator=g).to(dtype)


@pytest.mark.parametrize("D,Hq,Hkv,Sq,q_pos,split,chunks,causal,dtype,keys", [
    (128, 8, 2, 190, 0, None, [(190, 0)], True, torch.bfloat16, None),                    # tails in both dimensions
    (128, 4, 4, 512, 0, None, [(512, 0)], True, torch.bfloat16, None),                    # one q head per kv head: q tiles shared
    (128, 6, 2, 300, (40, 700), 130, [(128, 0), (77, 500), (256, 2000)], True, torch.bfloat16, None),  # a chunk no row sees
    (64, 8, 1, 200, 0, None, [(129, 0)], False, torch.bfloat16, None),
    (64, 8, 1, 1100, 0, None, [(300, 0)], False, torch.bfloat16, 256),                    # two 32-key halves per wave
    (64, 4, 2, 130, 64, None, [(64, 0), (200, 64)], True, torch.float32, None),
    (128, 4, 1, 333, 0, None, [(333, 0)], True, torch.float32, None),
])
def test_shared_key_tiles(ltr, D, Hq, Hkv, Sq, q_pos, split, chunks, causal, dtype, keys):
    from lightron_amd import _lib as L
    g = torch.Generator().manual_seed(D + Sq)
    B, f32 = 2, dtype == torch.float32
    q, do = (_randn((B, Sq, Hq, D), g, dtype).cuda() for _ in range(2))
    total = sum(n for n, _ in chunks)
    k, v = (_randn((B, total, Hkv, D), g, dtype).cuda() for _ in range(2))
    at = [sum(n for n, _ in chunks[:i]) for i in range(len(chunks))]
    cut = lambda t: [t[:, a:a + n] for a, (n, _) in zip(at, chunks)]
    pos = [p for _, p in chunks]
    o, lse = ltr.attn_fwd(q, cut(k), cut(v), pos, q_pos, split, causal)
    delta = ltr.attn_delta(o, do)
    seen = []
    real = L.load().ltr_attn_bwd_workspace

    def grads(share, out):
        dq = torch.zeros(q.shape, dtype=torch.float32, device="cuda")
        dk, dv = (torch.full(k.shape, 0.25, dtype=out, device="cuda") for _ in range(2))
        ltr.attn_bwd_accumulate(q, do, lse, delta, cut(k), cut(v), pos, dq, cut(dk), cut(dv), q_pos, split, causal, dkdv_keys=keys, share_keys=share)
        return dk, dv

    a = L.BwdArgs()
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.n_chunks = B, Hq, Hkv, D, Sq, len(chunks)
    qp = q_pos if isinstance(q_pos, tuple) else (q_pos, q_pos)
    a.q_pos0[0], a.q_pos0[1], a.q_split = qp[0], qp[1], Sq if split is None else split
    a.flags, a.io_dtype = (L.LTR_CAUSAL if causal else 0) | (L.LTR_DKDV_KEYS_256 if keys == 256 else 0), L.LTR_F32 if f32 else L.LTR_BF16
    for i, (n, p) in enumerate(chunks):
        a.chunk[i].sk, a.chunk[i].pos0 = n, p
    want = ctypes.c_int64()
    assert real(ctypes.byref(a), ctypes.byref(want)) == 0 and want.value > 0      # the problem is one whose tiles are shared
    for out in ([torch.float32] if f32 else [torch.float32, torch.bfloat16]):
        plain, shared, again = grads(False, out), grads(True, out), grads(True, out)
        for x, y, z in zip(plain, shared, again):
            assert torch.equal(y, z)                                              # fixed order: reproducible
            # the same fp32 terms in another order; a bf16 result may round to the neighbour: 2^-8 of its own size
            err = (x.float() - y.float()).abs()
            bound = 1e-5 * x.float().abs().max() + (x.float().abs() / 128 if out == torch.bfloat16 else 0)
            assert (err <= bound).all()
    # and against the dense oracle (accumulators started at 1/4, bf16 results are written)
    dk, dv = grads(True, dtype)
    rows = torch.arange(Sq)
    qpos = rows + qp[0] if split is None else torch.where(rows < split, rows + qp[0], rows - split + qp[1])
    kpos = torch.cat([torch.arange(p, p + n) for n, p in chunks])
    ref = orc.dense_attention_grads(q.cpu().float(), k.cpu().float(), v.cpu().float(), do.cpu().float(), qpos, kpos, causal, dtype=torch.float32)
    for got, r in zip((dk, dv), ref[3:5]):
        got = got.cpu().float() - (0.25 if f32 else 0.0)
        assert (got - r).norm() <= (1e-4 if f32 else 5e-2) * r.norm()


@pytest.mark.parametrize("D,Hq,Hkv,dtype", [(128, 6, 2, torch.bfloat16), (64, 8, 1, torch.bfloat16), (64, 4, 1, torch.float32)])
def test_masked_tiles_between_shared_ones(ltr, D, Hq, Hkv, dtype):
    """Chunks and tails of chunks that no row sees lie before and between the visible ones of the table: they have no partial sums,
    and the visible tiles' partials are numbered without them."""
    test_shared_key_tiles(ltr, D, Hq, Hkv, 300, (40, 700), 130, [(300, 2000), (128, 0), (140, 3000), (520, 500), (77, 1500), (64, 128)], True, dtype, None)


@pytest.mark.parametrize("D,Hq,Hkv,S,causal", [(128, 4, 1, 1000, True), (64, 4, 2, 2000, False)])
def test_shared_fp32_sums_are_no_further_from_fp64(ltr, D, Hq, Hkv, S, causal):
    """fp32 sums of up to 4096 rows: several shorter ones added up have the smaller rounding error."""
    g = torch.Generator(device="cuda").manual_seed(S)
    q, do = (torch.randn(1, S, Hq, D, device="cuda", generator=g) for _ in range(2))
    k, v = (torch.randn(1, S, Hkv, D, device="cuda", generator=g) for _ in range(2))
    plan = ltr.attn_plan(1, Hq, Hkv, D, S, [S], [0], causal=causal, dtype=torch.float32, share_keys=True)["dkdv"]
    assert plan["blocks_per_tile"] > 1 and plan["reduce_blocks"] > 0
    o, lse = ltr.attn_fwd(q, [k], [v], [0], causal=causal)
    delta = ltr.attn_delta(o, do)
    want = [torch.zeros(k.shape, dtype=torch.float64, device="cuda") for _ in range(2)]
    for h in range(Hq):
        qh, doh, kh, vh = (t[0, :, i].double() for t, i in ((q, h), (do, h), (k, h * Hkv // Hq), (v, h * Hkv // Hq)))
        s = qh @ kh.T * D ** -0.5
        p = (s.masked_fill(~torch.ones(S, S, dtype=torch.bool, device="cuda").tril(), -torch.inf) if causal else s).softmax(-1)
        ds = p * (doh @ vh.T - (doh * (p @ vh)).sum(-1, keepdim=True)) * D ** -0.5
        want[0][0, :, h * Hkv // Hq] += ds.T @ qh
        want[1][0, :, h * Hkv // Hq] += p.T @ doh
    err = []
    for share in (False, True):
        got = [torch.zeros_like(k) for _ in range(2)]
        ltr.attn_bwd_accumulate(q, do, lse, delta, [k], [v], [0], torch.zeros_like(q), got[:1], got[1:], 0, None, causal, share_keys=share)
        err.append([((x.double() - w).norm() / w.norm()).item() for x, w in zip(got, want)])
    assert all(shared <= whole for whole, shared in zip(*err)) and max(err[1]) < 2e-6
    rows = 4097 * Hkv // Hq + 1          # and one row more than the rule takes: the whole sum
    assert ltr.attn_plan(1, Hq, Hkv, D, rows, [rows], [0], causal=causal, dtype=torch.float32, share_keys=True)["dkdv"]["blocks_per_tile"] == 1
