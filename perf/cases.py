"""The work that users of this package have it do, as cases that can be timed and compared: attention forward and backward
through the public entry points, from the smallest training call of the reference's default configuration (four sequences of
128 tokens) to a whole ring over 32768 tokens.

A case is a dict of plain values.  Its "kind" says which entry point a pass goes through:

  call     block_attention on one K/V chunk: the attention call of a transformer layer (training or forward only).
  ring     ring_attention_kernel as ONE rank of a ring: its Q chunk against the K/V chunks of all ranks, resident on the
           GPU; stepwise = one launch per ring step, as when the chunks arrive one at a time.
  rings    ring_attention_kernel for ALL ranks of a ring, dK / dV summed over the ranks in the ring's fp32 accumulators.
  ulysses  the sequence -> head exchange of q, k, v (rank-stacked), full attention on the local heads, and back.
  layer    ContextParallelAttention around Attention (ranks > 1) or Attention alone (ranks = 1): projections, RoPE,
           attention and output projection, with the gradients of the input and of the weights.

B, Hq, Hkv, D: batch, query heads, key/value heads, head dim.  S: tokens of the whole sequence; ranks: over how many ranks
it is cut (call: 1).  data: "normal" = N(0, 1), "half" = N(0, 1) / 2, "uniform" = U(-1, 1), "rope" = N(0, 1) with RoPE
applied to q and k beforehand."""
import math
from types import SimpleNamespace

import torch

import lightron_amd as la
from lightron_amd.parallel_cp import _all_to_all

TYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(kind, B, Hq, Hkv, D, S, ranks=1, rank=0, causal=True, train=True, dtype="bf16", layout="contiguous", stepwise=False,
          data="normal", name=None):
    c = dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, S=S, ranks=ranks, rank=rank, causal=causal, train=train, dtype=dtype,
             layout=layout, stepwise=stepwise, data=data)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the reference's default training call: micro-batch 4, 12 heads of 64, 128 tokens; latency and launches count
        _case("call", 4, 12, 12, 64, 128, name="call_s128"),
        # the same model at its full context and an ordinary batch
        _case("call", 16, 12, 12, 64, 1024, name="call_s1024"),
        # attention of a large layer, one chunk, head dim 128
        _case("call", 8, 32, 32, 128, 2048, name="call_s2048"),
        # a single sequence of odd length with grouped heads: few query rows, nothing a multiple of a tile
        _case("call", 1, 32, 8, 128, 1237, name="call_gqa_s1237"),
        # a head dim that has no kernel of its own, odd length
        _case("call", 2, 16, 16, 96, 777, name="call_d96_s777"),
        # the reference's acceptance dtype: four ranks of 256 tokens in fp32, trained
        _case("rings", 2, 8, 8, 64, 1024, ranks=4, dtype="fp32", name="rings_fp32_s1024"),
        # forward of the last rank of a ring: 1024 tokens against 8 chunks
        _case("ring", 4, 32, 32, 128, 8192, ranks=8, rank=7, train=False, data="half", name="ring_fwd_s8192"),
        # the headline: a whole ring of eight zig-zag shares over 32768 tokens, grouped heads, trained
        _case("rings", 1, 32, 8, 128, 32768, ranks=8, layout="zigzag", name="rings_zigzag_s32768"),
        # one rank of that ring in the call pattern of a real ring, one launch per step
        _case("ring", 1, 32, 8, 128, 32768, ranks=8, rank=0, layout="zigzag", stepwise=True, name="ring_stepwise_s32768"),
        # long context: the last of 16 ranks over 131072 tokens, RoPE applied beforehand
        _case("ring", 1, 8, 8, 128, 131072, ranks=16, rank=15, data="rope", name="ring_s131072"),
        # Ulysses layout: exchange, full attention on the local heads, exchange back, for all four ranks
        _case("ulysses", 8, 16, 16, 64, 4096, ranks=4, causal=False, data="uniform", name="ulysses_s4096"),
        # a context-parallel attention layer with its projections and RoPE
        _case("layer", 1, 16, 16, 128, 4096, ranks=4, name="layer_cp4_s4096"),
    ]


def _cost(c):
    """Rough time of a pass in units of bf16 matrix work: what keeps drawn cases below the largest listed one."""
    slow = (12 if c["dtype"] == "fp32" else 1) * (1 if c["D"] in (64, 128) else 3) * (2 if c["D"] == 64 else 1)
    return slow * work(c)["flops"]


def draw(rng):
    def log_size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["call", "call", "call", "ring", "ring", "rings", "ulysses", "layer"])
    heads = rng.choice([(8, 8), (12, 12), (16, 16), (16, 4), (32, 8), (32, 32)])
    D = rng.choice([64, 128, 128, 64, 128, 64, 96, 80]) if kind == "call" else rng.choice([64, 128])
    B = log_size(1, 16)
    dtype = "fp32" if kind in ("call", "ring", "rings") and rng.random() < 0.15 else "bf16"
    train = rng.random() < 0.75 or kind == "rings"
    if kind == "call":
        c = _case(kind, B, *heads, D, log_size(64, 16384), causal=rng.random() < 0.8, train=train, dtype=dtype)
    elif kind in ("ring", "rings"):
        ranks = rng.choice([2, 4, 8])
        layout = rng.choice(["contiguous", "zigzag"])
        local = 2 * log_size(32, 8192 if kind == "ring" else 2048)
        c = _case(kind, B, *heads, D, local * ranks, ranks=ranks, rank=rng.randrange(ranks), causal=layout == "zigzag" or rng.random() < 0.8,
                  train=train, dtype=dtype, layout=layout, stepwise=rng.random() < 0.4)
    elif kind == "ulysses":
        ranks = rng.choice([2, 4])
        c = _case(kind, B, heads[0], heads[0], D, log_size(32, 2048) * ranks, ranks=ranks, causal=rng.random() < 0.5, train=train, data="uniform")
    else:
        ranks = rng.choice([1, 1, 2, 4])
        c = _case(kind, B, *heads, D, log_size(32, 2048) * ranks, ranks=ranks, train=train)
    while _cost(c) > 1.5e13 or c["B"] * c["S"] * c["Hq"] * c["D"] > 1 << 28:
        if c["B"] > 1:
            c["B"] = (c["B"] + 1) // 2
        else:
            unit = 2 * c["ranks"]
            c["S"] = max(unit, c["S"] // 2 // unit * unit)
    return c


def _positions(c, r):
    """First positions of rank r's two segments and the segment length (contiguous: one segment of the whole share)."""
    W, n = c["ranks"], c["S"] // c["ranks"]
    return [(r * n, n)] if c["layout"] == "contiguous" else [(r * (n // 2), n // 2), ((2 * W - 1 - r) * (n // 2), n // 2)]


def _pairs(c, ranks):
    """Visible (query, key) pairs of the given ranks' queries against the whole sequence, per batch entry and head."""
    S = c["S"]
    if not c["causal"]:
        return len(ranks) * (S // c["ranks"]) * S
    return sum(n * p + n * (n + 1) // 2 for r in ranks for p, n in _positions(c, r))


def work(case):
    c = case
    e = 4 if c["dtype"] == "fp32" else 2
    all_ranks = c["kind"] in ("rings", "ulysses", "layer")
    rows = c["B"] * c["S"] // (1 if all_ranks else c["ranks"])
    q, kv, lse = rows * c["Hq"] * c["D"] * e, c["B"] * c["S"] * c["Hkv"] * c["D"] * e, rows * c["Hq"] * 4
    pairs = c["B"] * c["Hq"] * _pairs(c, range(c["ranks"]) if all_ranks else [c["rank"]])
    flops = (14 if c["train"] else 4) * c["D"] * pairs
    if c["kind"] == "layer":
        dim = c["Hq"] * c["D"]
        weights = dim * dim * 2 + dim * c["Hkv"] * c["D"] * 2
        tokens = c["B"] * c["S"]
        return {"bytes": (2 if c["train"] else 1) * (2 * tokens * dim + weights) * e,
                "flops": flops + (6 if c["train"] else 2) * tokens * weights}
    # forward: q, k, v in, O and LSE out; training: dO in, dQ, dK, dV out as well
    return {"bytes": 2 * q + 2 * kv + lse + (2 * q + 2 * kv if c["train"] else 0), "flops": flops}


def tolerance(case):
    # Four times the distance from float64 attention (layer) on the same inputs: relative 2.0e-3 .. 3.1e-3 in bf16 (O, dQ, dK, dV;
    # largest single difference 0.14, a bf16 gradient near zero), 6.2e-3 through the layer's four bf16 projections, and up to
    # 6e-7 in fp32 at 256 keys (1e-6 where the sums are some thousand terms long; largest 8e-6).
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 1e-4}
    return {"rel": 2.4e-2 if case["kind"] == "layer" else 1.2e-2, "max": 0.4}


def prepare(case, seed):
    c = case
    dev, dt = torch.device("cuda"), TYPES[c["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    B, Hq, Hkv, D, S, W = (c[k] for k in ("B", "Hq", "Hkv", "D", "S", "ranks"))
    n = S // W

    def tensor(*shape):
        if c["data"] == "uniform":
            x = torch.rand(*shape, generator=gen, device=dev) * 2 - 1
        else:
            x = torch.randn(*shape, generator=gen, device=dev)
        return (x * 0.5 if c["data"] == "half" else x).to(dt)

    def leaf(t):
        return t.requires_grad_(c["train"])

    s = SimpleNamespace(case=dict(c))
    if c["kind"] == "call":
        s.q, s.k, s.v = (leaf(tensor(B, S, h, D)) for h in (Hq, Hkv, Hkv))
        s.do = tensor(B, S, Hq, D)
    elif c["kind"] in ("ring", "rings"):
        mine = list(range(W)) if c["kind"] == "rings" else [c["rank"]]
        qs, kv = [tensor(B, n, Hq, D) for _ in mine], [(tensor(B, n, Hkv, D), tensor(B, n, Hkv, D)) for _ in range(W)]
        if c["data"] == "rope":
            freqs = la.precompute_freqs_cis(D, S, device=dev)
            at = [torch.cat([freqs[p:p + m] for p, m in _positions(c, r)]) for r in range(W)]
            kv = [(la.apply_rotary_emb(k, k, at[r])[0], v) for r, (k, v) in enumerate(kv)]
            qs = [la.apply_rotary_emb(q, q, at[r])[0] for q, r in zip(qs, mine)]
        s.qs, s.dos = [leaf(q) for q in qs], [tensor(B, n, Hq, D) for _ in mine]
        s.kv = [(leaf(k), leaf(v)) for k, v in kv]
        # all ranks of a ring, or a rank whose chunks travel on: fp32 accumulators that belong to the chunks
        s.acc = la.RingKVGrads(s.kv) if c["train"] and (c["kind"] == "rings" or c["stepwise"]) else None
        s.rings = [la.LocalRing(r, W, s.kv, causal=c["causal"], layout=c["layout"], stepwise=c["stepwise"], kv_grads=s.acc) for r in mine]
    elif c["kind"] == "ulysses":
        s.group = la.LocalCPGroup(W)
        s.q, s.k, s.v = (leaf(tensor(W, B, n, Hq, D)) for _ in range(3))
        s.do = tensor(W, B, n, Hq, D)
    else:
        dim = Hq * D
        args = SimpleNamespace(dim=dim, n_heads=Hq, n_kv_heads=Hkv, tp_size=1)
        with torch.device(dev):
            inner = la.Attention(args).to(dt)
        for p in inner.parameters():
            p.data.normal_(0, dim ** -0.5, generator=gen)
        s.layer = inner if W == 1 else la.ContextParallelAttention(inner, args, cp_group=la.LocalCPGroup(W))
        s.freqs = la.precompute_freqs_cis(D, S, device=dev)
        s.x = leaf(tensor(*((B, S, dim) if W == 1 else (W, B, n, dim))))
        s.do = tensor(*s.x.shape)
    return s


def _grads(tensors):
    out = [t.grad for t in tensors]
    for t in tensors:
        t.grad = None
    return out


def run(state):
    s, c = state, state.case
    with torch.set_grad_enabled(c["train"]):
        if c["kind"] == "call":
            o, lse = la.block_attention(s.q, [s.k], [s.v], [0], causal=c["causal"])
            if not c["train"]:
                return o, lse
            o.backward(s.do)
            return (o.detach(), lse, *_grads([s.q, s.k, s.v]))
        if c["kind"] in ("ring", "rings"):
            if s.acc is not None:
                s.acc.zero_()
            outs = []
            for ring, q, do in zip(s.rings, s.qs, s.dos):
                k, v = s.kv[ring.rank]
                o = la.ring_attention_kernel(q, k, v, ring, None)
                if c["train"]:
                    o.backward(do)
                outs += [o.detach()] + ([] if c["train"] else [ring.last_lse])
            if not c["train"]:
                return outs
            outs += _grads(s.qs)
            if s.acc is not None:
                return outs + list(s.acc.finalize(assign=False))
            return outs + _grads([t for kv in s.kv for t in kv])
        if c["kind"] == "ulysses":
            W, B, n, H, D = s.q.shape
            q, k, v = (_all_to_all(t, 2, 1, s.group).reshape(W * B, W * n, H // W, D) for t in (s.q, s.k, s.v))
            o, _ = la.block_attention(q, [k], [v], [0], causal=c["causal"])
            o = _all_to_all(o.view(W, B, W * n, H // W, D), 1, 2, s.group)
            if not c["train"]:
                return o
            o.backward(s.do)
            return (o.detach(), *_grads([s.q, s.k, s.v]))
        o = s.layer(s.x, s.freqs)
        if not c["train"]:
            return o
        o.backward(s.do)
        return (o.detach(), *_grads([s.x, *s.layer.parameters()]))
