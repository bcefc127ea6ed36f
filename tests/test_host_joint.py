"""CPU tests of the backward in one launch (LTR_BWD_JOINT): the block order of its two kinds (csrc/ltr_blocks.h, compiled with the host
compiler), the launch times it is chosen by, and its plans."""
import ctypes
import heapq
import os
import random
import shutil
import subprocess
import time
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

import lightron_amd as la
from lightron_amd import _lib as L

CSRC = os.path.join(os.path.dirname(la.__file__), "csrc")
PROGRAM = r"""
#include "ltr_blocks.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
// "order" pairs q_items q_inner q_group kv_items kv_inner kv_group keys_first -> "ok"; "time" slots (us n)... -> launch_us, and whether the
// same comes of it in two parts, the second after a copy of the first, and what a limit says
int main(int argc, char **argv) {
    if (argv[1][0] == 't') {
        std::vector<BlockClass> c;
        for (int i = 3; i < argc; i += 2) c.push_back({atof(argv[i]), atoll(argv[i + 1])});
        const int k = (int)c.size(), slots = atoi(argv[2]);
        const double us = launch_us(c.data(), k, slots);
        bool same = true;
        for (int cut = 0; cut <= k; cut++) {
            Dispatch first(slots);
            first.add(c.data(), cut);
            for (int again = 0; again < 2; again++) {
                Dispatch d(first);
                same = same && d.add(c.data() + cut, k - cut) && d.end == us;
            }
        }
        same = same && !Dispatch(slots).add(c.data(), k, us) && Dispatch(slots).add(c.data(), k, us * 1.0001);
        printf("%.6f %d\n", us, same);
        return 0;
    }
    long long a[10];
    for (int i = 2; i < argc; i++) a[i] = atoll(argv[i]);
    const int pairs = (int)a[2], keys_first = (int)a[9];
    const BlockMap m[2] = {block_grid(pairs, a[3], a[4], a[5]).map, block_grid(pairs, a[6], a[7], a[8]).map};
    const long long n[2] = {(long long)pairs * a[3] * a[4], (long long)pairs * a[6] * a[7]};
    const unsigned places[2] = {map_blocks(m[0], pairs), map_blocks(m[1], pairs)};
    const JointMap j = {places[keys_first], keys_first};
    std::vector<unsigned char> seen[2] = {std::vector<unsigned char>(n[0]), std::vector<unsigned char>(n[1])};
    long long got[2] = {};
    std::vector<int> order[2] = {std::vector<int>(8), std::vector<int>(8)};
    for (unsigned id = 0; id < places[0] + places[1]; id++) {
        const JointItem b = joint_item_at(j, m[0], m[1], pairs, id);
        const int kv = b.keys, items = (int)(kv ? a[6] : a[3]), inner = (int)(kv ? a[7] : a[4]);
        if ((id < j.first) != (b.keys == (keys_first != 0))) return printf("kind\n"), 1;
        if (b.item.pair >= pairs) continue;
        if (b.item.pair < 0 || b.item.item < 0 || b.item.item >= items || b.item.sub < 0 || b.item.sub >= inner) return printf("range\n"), 1;
        if (pairs % 8 == 0 && (b.item.pair & 7) != (int)(id & 7)) return printf("xcd\n"), 1;
        if (seen[kv][((long long)b.item.pair * items + b.item.item) * inner + b.item.sub]++) return printf("twice\n"), 1;
        got[kv]++;
    }
    if (got[0] != n[0] || got[1] != n[1]) return printf("missing\n"), 1;
    printf("ok\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = os.environ.get("CXX", "g++")
    if not shutil.which(cxx):
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("joint")
    (d / "joint.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", CSRC, str(d / "joint.cpp"), "-o", str(d / "joint")], check=True)
    return lambda *a: subprocess.run([str(d / "joint")] + [str(x) for x in a], capture_output=True, text=True).stdout.strip()


@pytest.mark.parametrize("pairs,q,kv", [
    (8, (1, 1, 1), (1, 1, 1)), (8, (5, 4, 1), (10, 4, 1)), (40, (7, 2, 5), (9, 1, 3)), (104, (3, 1, 7), (6, 2, 13)),   # last groups with empty places
    (7, (9, 4, 1), (5, 2, 1)), (1, (3, 8, 1), (2, 16, 1)), (12, (4, 3, 1), (1, 1, 1)),                                   # pairs that do not divide among the XCDs
])
@pytest.mark.parametrize("keys_first", [0, 1])
def test_every_block_of_both_kinds_once(program, pairs, q, kv, keys_first):
    assert program("order", pairs, *q, *kv, keys_first) == "ok"


def _dispatch(classes, slots):
    free, end = [0.0] * slots, 0.0
    for us, n in classes:
        for _ in range(n):
            t = heapq.heappop(free) + us
            end = max(end, t)
            heapq.heappush(free, t)
    return end


def test_launch_time_is_that_of_in_order_dispatch(program):
    """Against the slots one by one: times within 3 % of a block count as one, which moves the end by a few such steps at most."""
    rng = random.Random(3)
    for _ in range(60):
        slots = rng.choice([1, 7, 32, 256])
        classes = [(rng.uniform(2, 60), rng.randrange(1, 3 * slots + 2)) for _ in range(rng.randrange(1, 17))]
        want = _dispatch(classes, slots)
        got, same = program("time", slots, *[x for c in classes for x in c]).split()
        got = float(got)
        assert same == "1", (slots, classes)
        assert abs(got - want) <= 0.06 * max(us for us, _ in classes) + 0.02 * want, (slots, classes, got, want)


def _args(D, B, Hq, Hkv, Sq, chunks, flags, dtype=L.LTR_BF16, q_pos0=(0, 0), q_split=None):
    a = L.BwdArgs()
    a.B, a.Hq, a.Hkv, a.D, a.Sq, a.q_split, a.n_chunks, a.flags, a.io_dtype = B, Hq, Hkv, D, Sq, Sq if q_split is None else q_split, len(chunks), flags, dtype
    a.q_pos0 = (ctypes.c_int64 * 2)(*q_pos0)
    for i, (sk, pos0) in enumerate(chunks):
        a.chunk[i].sk, a.chunk[i].pos0 = sk, pos0
    return a


def test_only_with_the_flag_and_without_size_hints():
    case = dict(B=2, Hq=16, Hkv=16, D=128, Sq=600, chunk_lens=[600], k_pos0=[0], causal=True)
    both = la.attn_plan(**case, joint=True)
    assert both["dq"]["kernel"] == both["dkdv"]["kernel"] and both["dq"]["kernel"].startswith("bwd_joint_kernel<128, ")
    for kw in ({}, dict(share_keys=True), dict(joint=True, dq_rows=256), dict(joint=True, dkdv_keys=128), dict(joint=True, dtype=torch.float32)):
        p = la.attn_plan(**case, **kw)
        assert p["dq"]["kernel"] != p["dkdv"]["kernel"], kw
    f = L.LTR_BWD_JOINT | L.LTR_CAUSAL
    for skip in (L.LTR_NO_DQ, L.LTR_NO_DKDV):   # one kind of blocks only
        p = L.AttnPlan()
        assert L.load().ltr_attn_plan(ctypes.byref(_args(128, 2, 16, 16, 600, [(600, 0)], f | skip)), ctypes.byref(p)) == 0
        assert p.dq_kernel != p.dkdv_kernel


def test_plans_of_joint_launches_hold_together():
    """Workspace, blocks and rows of random problems belong to each other; past several rounds of blocks nothing is joined."""
    rng = random.Random(1)
    joint = own = 0
    for _ in range(400):
        n_rep, Hkv, D = rng.choice([1, 2, 4]), rng.choice([1, 4, 8, 12, 16]), rng.choice([64, 128, 96, 40])
        B, S, n, causal = rng.choice([1, 2, 5, 16]), rng.randrange(1, rng.choice([200, 5000])), rng.choice([1, 1, 3]), rng.random() < 0.7
        chunks = [(rng.randrange(1, S + 1), i * S) for i in range(n)]
        f = L.LTR_BWD_JOINT | L.LTR_HEAD_COLS | (L.LTR_CAUSAL if causal else 0) | rng.choice([0, L.LTR_DELTA_FROM_O | L.LTR_DQ_BF16 | L.LTR_DKDV_BF16])
        a = _args(D, B, n_rep * Hkv, Hkv, S, chunks, f)
        need, ws = ctypes.c_int64(0), L.AttnPlanWs()
        assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)) == 0
        assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value, ctypes.byref(ws)) == 0
        if ws.plan.dq_kernel != ws.plan.dkdv_kernel:
            continue
        joint += 1
        width = 64 if D <= 64 else 128
        pad = "" if D in (64, 128) else "_pad"
        if ws.plan.dq_kernel.startswith(b"bwd_joint_delta"):   # DELTA by the blocks themselves: few rows, one round, nothing given
            assert ws.plan.dq_kernel.decode() == "bwd_joint_delta%s_kernel<%d>" % (pad, width) and ws.plan.dq_rows == 128
            assert f & L.LTR_DELTA_FROM_O and S <= (320 if width == 64 else 144) and ws.plan.dq_blocks + ws.plan.dkdv_blocks <= 256
            own += 1
        else:
            assert ws.plan.dq_kernel.decode() == "bwd_joint%s_kernel<%d, %d>" % (pad, width, 256 // ws.plan.dq_rows)
        assert ws.plan.dq_rows in (128, 256) and not ws.plan.dq_paired and ws.plan.dkdv_keys == 128
        assert ws.plan.dq_blocks == -(-S // ws.plan.dq_rows) * B * n_rep * Hkv
        tiles = sum(-(-(min(sk, S - p) if causal else sk) // 128) for sk, p in chunks if not causal or p < S)
        t = ws.blocks_per_tile
        assert need.value == (tiles * B * Hkv * t * 128 * width * 8 if t > 1 else 0)
        assert ws.plan.dkdv_blocks == (tiles if t > 1 else sum(-(-sk // 128) for sk, _ in chunks)) * B * Hkv * t
        if need.value:   # one byte short: no shared tiles
            assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value - 1, ctypes.byref(ws)) == 0 and ws.blocks_per_tile == 1
    assert joint > 100 and own > 3
    big = la.attn_plan(8, 32, 32, 128, 4096, [4096], [0], causal=True, joint=True)
    assert big["dq"]["kernel"] == "bwd_dq_kernel<128, 1>" and big["dkdv"]["kernel"] == "bwd_dkdv_kernel<128, 1>"


def test_the_plan_kept_is_that_of_the_problem():
    """A thread keeps plans: problems that differ in one number each, asked for in turn, in both orders and on several threads, and more of them
    than places."""
    base = dict(B=2, Hq=16, Hkv=4, D=128, Sq=700, chunks=[(700, 0), (300, 700)], flags=L.LTR_BWD_JOINT | L.LTR_CAUSAL | L.LTR_HEAD_COLS)
    variants = [base] + [dict(base, **kw) for kw in (dict(B=3), dict(Hq=8), dict(Hkv=16), dict(D=96), dict(Sq=900), dict(chunks=[(700, 0)]),
                                                     dict(chunks=[(700, 0), (301, 700)]), dict(chunks=[(700, 0), (300, 600)]),
                                                     dict(flags=base["flags"] & ~L.LTR_CAUSAL), dict(flags=base["flags"] | L.LTR_DELTA_FROM_O))]

    def ask(v):
        a, need, ws = _args(**v), ctypes.c_int64(0), L.AttnPlanWs()
        assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)) == 0
        assert L.load().ltr_attn_plan_ws(ctypes.byref(a), need.value, ctypes.byref(ws)) == 0
        p = ws.plan
        return need.value, ws.blocks_per_tile, p.dq_kernel, p.dkdv_kernel, p.dq_blocks, p.dkdv_blocks, p.dq_rows, p.fwd_rows, p.fwd_blocks, p.fwd_kernel

    # ranks of a ring differ in where their rows stand, and zig-zag shares from contiguous ones in where the rows are cut: other key tiles are seen
    ring = dict(base, Sq=512, chunks=[(256, i * 256) for i in range(8)], q_pos0=(256, 256), q_split=256)
    ranks = [ring, dict(ring, q_pos0=(256, 1024)), dict(ring, q_pos0=(1536, 256)), dict(ring, q_split=128), dict(ring, q_split=128, q_pos0=(256, 1024))]
    assert len({ask(v)[5] for v in ranks}) == len(ranks), [ask(v) for v in ranks]
    variants += ranks
    alone = [ask(v) for v in variants]
    assert len(set(alone)) > 6 + len(ranks)
    # a problem with its workspace and without one
    a, ws = _args(**base), L.AttnPlanWs()
    for need, shared in ((alone[0][0], True), (0, False), (alone[0][0], True)):
        assert alone[0][0] > 0 and L.load().ltr_attn_plan_ws(ctypes.byref(a), need, ctypes.byref(ws)) == 0 and (ws.blocks_per_tile > 1) == shared
    for order in (range(len(variants)), reversed(range(len(variants)))):
        for i in order:
            assert ask(variants[i]) == alone[i] == ask(variants[i])
    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(ask, variants * 20)) == alone * 20
    many = [dict(base, Sq=S, chunks=[(S, 0)]) for S in range(130, 130 * 121, 130)]   # one key tile more each

    def ask_anew(v):   # on a thread of its own, which keeps nothing yet
        with ThreadPoolExecutor(1) as one:
            return one.submit(ask, v).result()

    new = [ask_anew(v) for v in many]
    assert len(set(new)) == len(many) and [ask(v) for v in many] == new == [ask(v) for v in many]


def test_a_new_problem_is_priced_once():
    """Calls of a length not seen before, 8 heads of 128 and 8000 tokens: the launch takes the plan that the workspace was asked for, also where
    that plan needs none (query alone, query and launch: 6 and 10 us, for 10 and 24)."""
    need, ws = ctypes.c_int64(0), L.AttnPlanWs()
    flags = L.LTR_CAUSAL | L.LTR_DELTA_FROM_O | L.LTR_DQ_BF16 | L.LTR_DKDV_BF16 | L.LTR_BWD_JOINT | L.LTR_FWD_ROWS_256   # the forward is given
    call = lambda S: ctypes.byref(_args(128, 1, 8, 8, S, [(S, 0)], flags))
    query = lambda r: L.load().ltr_attn_bwd_workspace(r, ctypes.byref(need))

    def both(r):
        query(r)
        L.load().ltr_attn_plan_ws(r, 0, ctypes.byref(ws))

    lengths = {query: range(8000, 8200), both: range(8200, 8400)}
    for S in (*lengths[query], *lengths[both]):
        query(call(S))
        assert need.value == 0
    best = {query: 1e9, both: 1e9}
    for lap in range(100):   # in turn, so that a busy machine is busy for both; more lengths than a thread keeps plans
        for ask in best:
            calls = [call(S) for S in lengths[ask][lap % 7::7]]
            start = time.perf_counter()
            for r in calls:
                ask(r)
            best[ask] = min(best[ask], (time.perf_counter() - start) / len(calls) * 1e6)
    assert best[both] < 2 * best[query], best


def test_the_plan_does_not_depend_on_what_was_asked_before():
    """Where the workspace query says 0 bytes the launch's plan is the same whether or not the query came first."""
    rng = random.Random(7)
    zero = 0

    def fresh(a, query):   # on a thread that has kept nothing
        def ask():
            need, ws = ctypes.c_int64(0), L.AttnPlanWs()
            if query:
                assert L.load().ltr_attn_bwd_workspace(ctypes.byref(a), ctypes.byref(need)) == 0
            assert L.load().ltr_attn_plan_ws(ctypes.byref(a), 0, ctypes.byref(ws)) == 0
            p = ws.plan
            return need.value, (ws.blocks_per_tile, p.dq_kernel, p.dkdv_kernel, p.dq_blocks, p.dkdv_blocks, p.dq_rows)
        with ThreadPoolExecutor(1) as one:
            return one.submit(ask).result()

    for _ in range(150):
        n_rep, Hkv, D, S = rng.choice([1, 2, 4]), rng.choice([1, 4, 8, 12]), rng.choice([64, 128, 96]), rng.randrange(60, 5000)
        a = _args(D, rng.choice([1, 2, 4]), n_rep * Hkv, Hkv, S, [(S, 0)], L.LTR_BWD_JOINT | L.LTR_HEAD_COLS | (L.LTR_CAUSAL if rng.random() < 0.7 else 0))
        need, asked = fresh(a, True)
        assert asked == fresh(a, False)[1]
        zero += need == 0
    assert zero > 30
