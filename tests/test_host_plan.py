"""CPU tests of the launch plans: head dims that run in the next width's kernels, and key tiles shared with a workspace."""
import ctypes
import random
import re
import shutil
import subprocess

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


def _kernels_of_the_library():
    """Demangled names of the kernels compiled into the library, as a profiler shows them."""
    out = subprocess.run(["nm", "-C", la._lib.LIB_PATH], capture_output=True, text=True, check=True).stdout
    return set(re.findall(r"(?:\(anonymous namespace\)::|\s)(\w+_kernel<[^()]*>)\(", out.replace("__device_stub__", "")))


@pytest.mark.skipif(shutil.which("nm") is None, reason="no nm")
def test_every_plan_names_kernels_that_exist():
    names = _kernels_of_the_library()
    assert "bwd_dkdv_reduce_kernel<64, 1>" in names
    rng = random.Random(5)
    seen = set()
    for _ in range(400):
        D = rng.choice([40, 64, 64, 96, 128, 128])
        dtype = rng.choice([torch.bfloat16, torch.float32]) if D in (64, 128) else torch.bfloat16
        Hkv, rep, B, Sq = rng.choice([1, 4, 8, 12, 16]), rng.choice([1, 2, 4]), rng.choice([1, 2, 5, 8, 32]), rng.choice([1, 16, 100, 256, 777, 1024, 2048, 4096])
        lens = rng.choice([[Sq], [128, 300], [2048] * 4])
        plan = la.attn_plan(B, Hkv * rep, Hkv, D, Sq, lens, [sum(lens[:i]) for i in range(len(lens))], 0, None, rng.random() < 0.7, dtype=dtype, share_keys=rng.random() < 0.5)
        for k in (plan["fwd"]["kernel"], plan["dq"]["kernel"], plan["dkdv"]["kernel"], plan["dkdv"].get("reduce_kernel", "")):
            assert k == "" or k in names, k
            seen.add(k)
    for part in ("w4", "shares", "pad", "keywave", "f32_mfma_kernel<64, 4>", "f32_rows32_kernel<64, 4>", "f32_mfma_kernel<128, 2>", "reduce"):
        assert any(part in k for k in seen), part


@pytest.mark.parametrize("pairs,Sq,kernel,rows", [
    (16, 256, "f32_mfma_kernel<64, 4>", 16), (16, 257, "f32_rows32_kernel<64, 4>", 32), (1, 4096, "f32_mfma_kernel<64, 4>", 16),
    (1, 4097, "f32_rows32_kernel<64, 4>", 32), (64, 512, "f32_mfma_kernel<64, 1>", 128), (33, 512, "f32_mfma_kernel<64, 2>", 64),
])
def test_fp32_rows_and_names_belong_together(pairs, Sq, kernel, rows):
    """Groups of 16 rows and of 32 rows with four key shares are different kernels: a name stands for one of them."""
    plan = la.attn_plan(1, pairs, pairs, 64, Sq, [64], [0], 0, None, True, dtype=torch.float32)
    assert plan["compute_units"] != 256 or (plan["fwd"]["kernel"], plan["fwd"]["rows"]) == ("fwd_" + kernel, rows)
    assert plan["compute_units"] != 256 or (plan["dq"]["kernel"], plan["dq"]["rows"]) == ("bwd_dq_" + kernel, rows)


@pytest.mark.parametrize("B,Hq,Hkv,S", [(8, 32, 32, 1024), (16, 16, 4, 700), (8, 16, 16, 2048), (8, 32, 8, 1100), (8, 32, 32, 512)])
def test_a_chunk_table_takes_the_kernels_of_one_chunk(B, Hq, Hkv, S):
    """The same rows and keys in one chunk or in two are the same work: at head dim 64 four-wave blocks, also where the pairs of 256-row
    tiles fill whole rounds of CUs."""
    one, two = (la.attn_plan(B, Hq, Hkv, 64, S, lens, pos, 0, None, True) for lens, pos in (([S], [0]), ([256, S - 256], [0, 256])))
    assert one == two
    assert one["compute_units"] != 256 or one["fwd"]["kernel"] == "fwd_bf16_w4_kernel<64>"


@pytest.mark.parametrize("lens", [[2048], [1024, 1024]])
def test_one_round_of_pairs_at_head_dim_64(lens):
    """4 x 16 heads of 2048 rows: 256 equal blocks of paired tiles against four blocks per CU of which three run at once (50 and 53 us)."""
    plan = la.attn_plan(4, 16, 16, 64, 2048, lens, [0, 1024][:len(lens)], 0, None, True)
    if plan["compute_units"] == 256:
        assert plan["fwd"]["kernel"] == "fwd_bf16_kernel<64, 1>" and plan["fwd"]["paired"] and plan["fwd"]["blocks"] == 256
    wider = la.attn_plan(8, 16, 16, 64, 1024, [1024], [0], 0, None, True)   # modelled 7 % shorter, measured 3 %
    assert wider["compute_units"] != 256 or wider["fwd"]["kernel"] == "fwd_bf16_w4_kernel<64>"


@pytest.mark.parametrize("B,Hq,Hkv,S", [(8, 16, 4, 135), (8, 16, 4, 200), (4, 32, 32, 164), (8, 16, 16, 252)])
def test_one_round_of_shares_stays(B, Hq, Hkv, S):
    """256 blocks of 128 rows against 128 blocks of 256 (12 and 16 us): every CU has a block."""
    plan = la.attn_plan(B, Hq, Hkv, 128, S, [S], [0], 0, None, True)
    if plan["compute_units"] == 256:
        assert plan["fwd"]["kernel"] == "fwd_bf16_shares_kernel<128, 2>" and plan["dq"]["kernel"] == "bwd_dq_shares_kernel<128, 2>"


@pytest.mark.parametrize("B,Hq,Hkv,S,causal", [(1, 1, 1, 500, True), (1, 2, 1, 200, False), (1, 2, 1, 500, True), (4, 32, 8, 1000, True), (1, 8, 4, 2000, False)])
def test_a_workspace_that_is_too_small_is_none(B, Hq, Hkv, S, causal):
    """Head dim 64, where shared key tiles take another kernel than tiles of one block: one byte short is the launch without a workspace."""
    a = _args(64, B, Hq, Hkv, S, [(S, 0)], L.LTR_CAUSAL if causal else 0)
    need, short, full = ctypes.c_int64(0), L.AttnPlanWs(), L.AttnPlanWs()
    assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)) == 0 and need.value > 0
    assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value - 1, ctypes.byref(short)) == 0
    assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value, ctypes.byref(full)) == 0 and full.blocks_per_tile > 1
    assert bytes(short.plan) == bytes(_plan(a)[1]) and short.blocks_per_tile == 1
