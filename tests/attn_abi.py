"""One backward through the C ABI with the flags given, for tests that need a kernel which block_attention's backward does not ask for (padded
heads without LTR_BWD_JOINT, accumulators at padded heads), and the plan that this very call has."""
import ctypes
from types import SimpleNamespace

import torch

from lightron_amd import _lib as L


def backward(q, do, o, lse, ks, vs, k_pos0, q_pos0=0, q_split=None, causal=False, joint=False, results=torch.bfloat16, fill=0.0, delta=None, share=True):
    """dq, dk, dv (results: bf16 receives them, fp32 adds to `fill`) and delta, from q, do, o [B, Sq, Hq, D] and chunks ks, vs; delta given: it is
    read, else the library writes it from o.  share: with the workspace that the library asks for."""
    B, Sq, Hq, D = q.shape
    a = L.BwdArgs()
    dq = torch.full(q.shape, fill, dtype=results, device=q.device)
    total = [sum(k.shape[1] for k in ks[:i]) for i in range(len(ks) + 1)]
    dk, dv = (torch.full((B, total[-1], ks[0].shape[2], D), fill, dtype=results, device=q.device) for _ in range(2))
    given = delta is not None
    if not given:
        delta = torch.full(lse.shape, 3.0, dtype=torch.float32, device=q.device)
    for name, t in (("q", q), ("d_o", do), ("lse", lse), ("delta", delta), ("dq", dq), ("o", o)):
        setattr(a, name, t.data_ptr())
    for name, t in (("q", q), ("do", do), ("dq", dq), ("k", ks[0]), ("v", vs[0]), ("dk", dk), ("dv", dv), ("o", o)):
        setattr(a, name + "_stride", (ctypes.c_int64 * 3)(*t.stride()[:3]))
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.n_chunks = B, Hq, ks[0].shape[2], D, Sq, len(ks)
    a.q_pos0 = (ctypes.c_int64 * 2)(*(q_pos0 if isinstance(q_pos0, tuple) else (q_pos0, q_pos0)))
    a.q_split = Sq if q_split is None else q_split
    a.scale, a.io_dtype = D ** -0.5, L.LTR_BF16
    a.flags = ((L.LTR_CAUSAL if causal else 0) | (L.LTR_HEAD_COLS if D not in (64, 128) else 0) | (L.LTR_BWD_JOINT if joint else 0)
               | (0 if given else L.LTR_DELTA_FROM_O) | (L.LTR_DQ_BF16 | L.LTR_DKDV_BF16 if results == torch.bfloat16 else 0))
    for i, (k, v) in enumerate(zip(ks, vs)):
        assert k.stride() == ks[0].stride() and v.stride() == vs[0].stride()
        c = a.chunk[i]
        c.k, c.v, c.dk, c.dv = k.data_ptr(), v.data_ptr(), dk[:, total[i]:].data_ptr(), dv[:, total[i]:].data_ptr()
        c.sk, c.pos0 = k.shape[1], k_pos0[i]
    lib, need, ws = L.load(), ctypes.c_int64(0), L.AttnPlanWs()
    if share:
        L.check(lib.ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)), "ltr_attn_bwd_workspace")
    L.check(lib.ltr_attn_plan_ws(ctypes.byref(a), need.value, ctypes.byref(ws)), "ltr_attn_plan_ws")
    part = torch.empty(need.value, dtype=torch.uint8, device=q.device) if need.value else None
    L.check(lib.ltr_attn_bwd_ws(ctypes.byref(a), None if part is None else part.data_ptr(), need.value, torch.cuda.current_stream().cuda_stream), "ltr_attn_bwd_ws")
    plan = SimpleNamespace(dq=ws.plan.dq_kernel.decode(), dkdv=ws.plan.dkdv_kernel.decode(), paired=bool(ws.plan.dq_paired), rows=ws.plan.dq_rows,
                           blocks=ws.plan.dq_blocks + ws.plan.dkdv_blocks, blocks_per_tile=ws.blocks_per_tile, keys_first=bool(ws.keys_first))
    return SimpleNamespace(dq=dq, dk=dk, dv=dv, delta=delta, plan=plan)
