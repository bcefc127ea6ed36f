"""CPU tests of the launch plans: head dims that run in the next width's kernels, and key tiles shared with a workspace."""
import ctypes

import pytest
import torch

import lightron_amd as la
from lightron_amd import _lib as L


def _args(D, B, Hq, Hkv, Sq, chunks, flags, dtype=L.LTR_BF16):
    a = L.BwdArgs()
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.q_split, a.n_chunks, a.flags, a.io_dtype = B, Hq, Hkv, D, Sq, Sq, len(chunks), flags, dtype
    for i, (sk, pos0) in enumerate(chunks):
        a.chunk[i].sk, a.chunk[i].pos0 = sk, pos0
    return a


def _plan(a):
    out = L.AttnPlan()
    return L.load().ltr_attn_plan(ctypes.byref(a), ctypes.byref(out)), out


def test_struct_of_the_workspace_plan():
    assert ctypes.sizeof(L.AttnPlanWs) == ctypes.sizeof(L.AttnPlan) + 8 + 8 + 48
    assert L.load().ltr_attn_plan_ws(None, 0, None) == -1
    assert L.load().ltr_attn_plan_ws(ctypes.byref(_args(64, 1, 4, 4, 64, [(64, 0)], 0)), -1, ctypes.byref(L.AttnPlanWs())) == -1


@pytest.mark.parametrize("D,width", [(8, 64), (56, 64), (72, 128), (96, 128), (120, 128)])
def test_head_cols_plan_names_the_padded_kernels(D, width):
    rc, pl = _plan(_args(D, 2, 16, 16, 777, [(777, 0)], L.LTR_CAUSAL | L.LTR_HEAD_COLS))
    assert rc == 0
    assert pl.fwd_kernel == b"fwd_bf16_pad_kernel<%d, %d>" % (width, 256 // pl.fwd_rows)
    assert pl.dq_kernel == b"bwd_dq_pad_kernel<%d, %d>" % (width, 256 // pl.dq_rows)
    assert pl.dkdv_kernel == b"bwd_dkdv_pad_kernel<%d>" % width and pl.dkdv_keys == 128
    assert _plan(_args(D, 2, 16, 16, 777, [(777, 0)], L.LTR_CAUSAL))[0] == -2                               # not without the flag,
    assert _plan(_args(D, 2, 16, 16, 777, [(777, 0)], L.LTR_CAUSAL | L.LTR_HEAD_COLS, L.LTR_F32))[0] == -2  # and bf16 only, as the launches
    assert la.attn_plan(2, 16, 16, D, 777, [777], [0], causal=True)["fwd"]["kernel"] == pl.fwd_kernel.decode()


def test_head_cols_at_a_native_width_changes_nothing():
    """B=32, 16 heads of 64, S=4096, no mask: wide blocks for all three kernels, flag or not."""
    plans = [_plan(_args(64, 32, 16, 16, 4096, [(4096, 0)], f))[1] for f in (0, L.LTR_HEAD_COLS)]
    assert bytes(plans[0]) == bytes(plans[1])
    assert plans[0].fwd_rows == plans[0].dq_rows == 512 and plans[0].dkdv_keys == 256


@pytest.mark.parametrize("dtype,width", [(torch.bfloat16, "bwd_dkdv_reduce_kernel<128, 1>"), (torch.float32, "bwd_dkdv_reduce_kernel<128, 1>")])
def test_shared_key_tiles_are_in_the_plan(dtype, width):
    """A short sequence with grouped heads: with its workspace the launch has n blocks per visible tile and a reduction."""
    case = (1, 32, 8, 128, 500, [500, 300], [0, 4000])
    alone, shared = (la.attn_plan(*case, causal=True, dtype=dtype, share_keys=s)["dkdv"] for s in (False, True))
    assert alone == dict(kernel=shared["kernel"], keys=128, blocks=7 * 8)                 # four tiles and three that no row sees
    n = shared["blocks_per_tile"]
    assert n > 1 and shared["blocks"] == 4 * 8 * n
    assert shared["reduce_kernel"] == width and shared["reduce_blocks"] == 7 * 8 * 4
    a = _args(128, 1, 32, 8, 500, [(500, 0), (300, 4000)], L.LTR_CAUSAL, L.LTR_F32 if dtype == torch.float32 else L.LTR_BF16)
    need = ctypes.c_int64(0)
    assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)) == 0 and need.value == 4 * 8 * n * 128 * 128 * 2 * 4
    ws = L.AttnPlanWs()                                                                    # one byte short: the unshared launch
    assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value - 1, ctypes.byref(ws)) == 0
    assert ws.blocks_per_tile == 1 and ws.reduce_blocks == 0 and ws.reduce_kernel == b"" and ws.plan.dkdv_blocks == 7 * 8


def test_plan_of_a_problem_that_shares_nothing():
    d = la.attn_plan(8, 32, 32, 128, 2048, [2048], [0], causal=True, share_keys=True)["dkdv"]
    assert d["blocks_per_tile"] == 1 and d["reduce_kernel"] == "" and d["reduce_blocks"] == 0
