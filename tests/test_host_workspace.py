"""CPU tests of the workspace that ltr_attn_bwd_workspace asks for (partial dK / dV of blocks that share a key tile)."""
import ctypes

import pytest

from lightron_amd import _lib as L

CAP = 512e6     # the library's bound on partial sums


def _workspace(B, Hq, Hkv, D, Sq, chunks, causal, q_pos0=(0, 0), q_split=None, dtype=L.LTR_BF16):
    a = L.BwdArgs()
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.n_chunks = B, Hq, Hkv, D, Sq, len(chunks)
    a.q_pos0[0], a.q_pos0[1], a.q_split = q_pos0[0], q_pos0[1], Sq if q_split is None else q_split
    a.flags, a.io_dtype = L.LTR_CAUSAL if causal else 0, dtype
    for i, (sk, pos0) in enumerate(chunks):
        a.chunk[i].sk, a.chunk[i].pos0 = sk, pos0
    n = ctypes.c_int64(-1)
    assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("Hq,Hkv,W,n", [(16, 4, 8, 16384), (8, 1, 32, 4096), (32, 8, 8, 4096), (32, 2, 16, 8192)])
def test_masked_key_tiles_need_no_workspace(Hq, Hkv, W, n):
    """The first ranks of a causal ring see few of the table's keys: they ask for what the visible keys alone would need."""
    for r in (0, 1, W // 2):
        table = [(n, j * n) for j in range(W)]
        full = _workspace(1, Hq, Hkv, 128, n, table, True, (r * n, r * n))
        assert full == _workspace(1, Hq, Hkv, 128, n, table[:r + 1], True, (r * n, r * n)) and full <= CAP
        assert full == _workspace(1, Hq, Hkv, 128, n, table[::-1], True, (r * n, r * n))


def test_workspace_is_bounded_over_the_ranks_of_zigzag_rings():
    for D in (64, 128):
        for Hq, Hkv in ((8, 1), (16, 4), (32, 8)):
            for W, h in ((4, 8192), (16, 2048), (16, 300)):
                table = [c for j in range(W) for c in ((h, j * h), (h, (2 * W - 1 - j) * h))]
                for r in range(W):
                    assert _workspace(1, Hq, Hkv, D, 2 * h, table, True, (r * h, (2 * W - 1 - r) * h), h) <= CAP
