"""Drop-in for parallel/parallel_cp.py of the reference (Ulysses-style context parallelism)
on ONE GPU.

The reference exchanges sequence shards for head shards with dist.all_to_all
(parallel_cp.py:49-73).  Here one process stands in for all W ranks of the cp group: a
tensor that passes through `SeqAllToAll` carries a leading rank dimension of size W
(``x[r]`` is what rank r would hold) and the exchange is an index permutation on the device.
`scatter_dim` / `gather_dim` keep their per-rank meaning (they index ``x[r]``).  With
group=None or a one-rank group the op is the identity, as in the reference (:55-56, :82-83).
"""
from __future__ import annotations

import torch
import torch.nn as nn

from . import attention
from .attention import block_attention
from .layers import rope_one, rope_table

_PLAIN = (torch.Tensor, nn.Parameter)
_CUS = 256               # of an MI355X
_MAX_BWD_ROWS = 4096 * 64    # q rows of one backward launch: its lists of 64-row q tiles hold 4096

class LocalCPGroup:
    """Stand-in for the cp ProcessGroup: `world_size` ranks emulated by one process."""

    def __init__(self, world_size: int):
        if world_size < 1:
            raise ValueError("world_size must be >= 1")
        self.world_size = world_size

    def size(self) -> int:
        return self.world_size


def _world_size(group) -> int:
    if group is None:
        return 1
    if isinstance(group, LocalCPGroup):
        return group.world_size
    import torch.distributed as dist
    if dist.is_available() and dist.is_initialized() and dist.get_world_size(group) == 1:
        return 1
    raise NotImplementedError("SeqAllToAll: this build runs on one GPU and has no collectives; pass a "
                              "LocalCPGroup (rank-stacked tensors) instead of a multi-rank ProcessGroup")


def _exchange_node(x: torch.Tensor):
    """The C++ binding when it can move this tensor (a plain GPU tensor whose bytes are its values), else None: under tracing, a
    dispatch mode or a tensor subclass the exchange is the torch ops below, which those see."""
    if not x.is_cuda or x.is_conj() or x.is_neg() or type(x) not in _PLAIN or not attention.USE_CPP_NODE:
        return None
    if torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None or torch._C._len_torch_dispatch_stack():
        return None
    return attention._cpp_node()


def _exchange(x: torch.Tensor, scatter_dim: int, gather_dim: int, W: int) -> torch.Tensor:
    """x: [W_src, *shard].  out[i] = cat_j(split(x[j], scatter_dim)[i], gather_dim)
    (parallel_cp.py:65-73 for every rank i at once)."""
    if x.shape[0] != W:
        raise RuntimeError("rank-stacked tensor must have leading dim %d, got %s" % (W, tuple(x.shape)))
    nd = x.dim() - 1
    sd, gd = scatter_dim % nd, gather_dim % nd
    size = x.size(sd + 1)
    assert size % W == 0, f"Input dim {scatter_dim} size {size} not divisible by CP size {W}"   # :61-63
    node = _exchange_node(x)
    if node:
        return node.exchange(x, sd, gd, W, attention._stream_ptr(x.device))      # one pass of ltr_copy_strided
    y = x.unflatten(sd + 1, (W, size // W))      # [W_src, ..., W_dst, chunk, ...]
    y = y.movedim(sd + 1, 0)                     # [W_dst, W_src, *shard with chunk at sd]
    y = y.movedim(1, gd + 1)                     # W_src just before the gather dim
    return y.flatten(gd + 1, gd + 2).contiguous()


class SeqAllToAll(torch.autograd.Function):
    @staticmethod
    def forward(ctx, input_tensor, scatter_dim, gather_dim, group):
        ctx.scatter_dim, ctx.gather_dim, ctx.group = scatter_dim, gather_dim, group
        W = _world_size(group)
        if W == 1:
            return input_tensor
        return _exchange(input_tensor, scatter_dim, gather_dim, W)

    @staticmethod
    def backward(ctx, grad_output):
        # forward: scatter(dim1) -> exchange -> gather(dim2); backward swaps the dims (:75-96)
        W = _world_size(ctx.group)
        if W == 1:
            return grad_output, None, None, None
        return _all_to_all(grad_output, ctx.gather_dim, ctx.scatter_dim, ctx.group), None, None, None


def _all_to_all(input_, scatter_dim, gather_dim, group):
    W = _world_size(group)
    nd = input_.dim() - 1
    if W > 1 and nd > 0 and input_.shape[0] == W and input_.shape[scatter_dim % nd + 1] % W == 0:
        node = _exchange_node(input_)
        if node:      # forward and backward as a C++ autograd node
            return node.seq_all_to_all(input_, scatter_dim % nd, gather_dim % nd, W, attention._stream_ptr(input_.device))
    return SeqAllToAll.apply(input_, scatter_dim, gather_dim, group)


class ContextParallelAttention(nn.Module):
    """Wrapper with the reference's constructor and forward (parallel_cp.py:120-245).

    `local_attn_module` supplies wq / wk / wv / wo and n_heads; `args` supplies n_heads, dim
    and tp_size.  The reference finds its cp group in a global device mesh; here it is passed
    as `cp_group` (a LocalCPGroup).  Without one the wrapped module is called unchanged
    (:161-162).  With one, `x` is rank-stacked [W, B, S_local, Hidden] and so is the result.

    literal=True follows the reference step by step (three seq->head exchanges, RoPE on the
    global sequence, causal attention on [B, S, H/W, D], head->seq exchange).  The default
    path gives the same result without the exchanges, which cancel: the shards are attended as
    the one sequence they are, all heads in one launch, or each
    against the shards as the kernel's chunk table (_one_sequence).
    """

    def __init__(self, local_attn_module, args, cp_group=None, literal: bool = False, causal: bool = True):
        super().__init__()
        self.local_attn = local_attn_module
        self.num_heads = args.n_heads
        if hasattr(local_attn_module, "n_heads"):
            self.num_heads = local_attn_module.n_heads
        else:
            self.num_heads = args.n_heads // getattr(args, "tp_size", 1)
        self.num_kv_heads = getattr(local_attn_module, "n_kv_heads", None) or self.num_heads
        self.head_dim = args.dim // args.n_heads
        self.cp_group = cp_group
        self.literal, self.causal = literal, causal
        if cp_group is not None:
            W = _world_size(cp_group)
            assert self.num_heads % W == 0, \
                f"Context Parallelism requires local_num_heads ({self.num_heads}) to be divisible by cp_size ({W})."

    def forward(self, x, freqs_cis):
        if self.cp_group is None:
            return self.local_attn(x, freqs_cis)
        W = _world_size(self.cp_group)
        if x.dim() != 4 or x.shape[0] != W:
            raise RuntimeError("with a LocalCPGroup x must be rank-stacked [W, B, S_local, Hidden]")
        _, B, S_local, _ = x.shape
        S_global = S_local * W
        assert freqs_cis.shape[0] >= S_global, f"freqs_cis too short: {freqs_cis.shape[0]} < S_global {S_global}"
        H, Hkv, D = self.num_heads, self.num_kv_heads, self.head_dim
        fc = freqs_cis[:S_global]
        if self.literal:
            xq = self.local_attn.wq(x).view(W, B, S_local, H, D)
            xk = self.local_attn.wk(x).view(W, B, S_local, Hkv, D)
            xv = self.local_attn.wv(x).view(W, B, S_local, Hkv, D)
            if Hkv % W:
                raise RuntimeError("literal Ulysses path needs n_kv_heads divisible by the cp size")
            xq = _all_to_all(xq, 2, 1, self.cp_group)            # [W, B, S_global, H/W, D]
            xk = _all_to_all(xk, 2, 1, self.cp_group)
            xv = _all_to_all(xv, 2, 1, self.cp_group)
            qf, kf, vf = (t.reshape(W * B, S_global, -1, D) for t in (xq, xk, xv))
            qf, kf = rope_one(qf, fc), rope_one(kf, fc)          # one streaming pass per tensor (q and k may differ in heads)
            o, _ = block_attention(qf, [kf], [vf], [0], 0, None, self.causal)
            o = o.view(W, B, S_global, H // W, D)
            o = _all_to_all(o, 1, 2, self.cp_group)              # [W, B, S_local, H, D]
            return self.local_attn.wo(o.flatten(3))
        if not self._one_sequence(x, S_global):
            return self._per_shard(x, fc)
        # The shards follow each other in the sequence, so the ranks' work is one attention over all of it: one launch per
        # kernel instead of one per shard (whose dK / dV autograd would have to add up).  RoPE at global positions (:215-219): K
        # in one streaming pass; q inside the attention kernel, dQ rotated back in the dQ kernel's epilogue (bf16; fp32 inputs
        # take the streaming pass for q as well)
        xs = x.transpose(0, 1).reshape(B, S_global, -1)
        xq = self.local_attn.wq(xs).view(B, S_global, H, D)
        xk = rope_one(self.local_attn.wk(xs).view(B, S_global, Hkv, D), fc)
        xv = self.local_attn.wv(xs).view(B, S_global, Hkv, D)
        fused = xq.dtype == torch.bfloat16
        o, _ = block_attention(xq if fused else rope_one(xq, fc), [xk], [xv], [0], 0, None, self.causal,
                               q_rope=rope_table(fc, xq.device) if fused else None)
        y = self.local_attn.wo(o.reshape(B, S_global, -1))
        return y.view(B, W, S_local, -1).transpose(0, 1).contiguous()

    def _one_sequence(self, x, S_global) -> bool:
        """Whether the shards are attended as one sequence, or one launch per shard against the shards as KV chunks.

        With one batch entry the shards are that sequence in memory already.  With more, joining them and splitting the result
        are two passes over the activations where per-shard launches pay one (their outputs are stacked).  In training the
        fewer launches and the dK / dV that need no adding up always pay for it (0.48 - 1.00 of the per-shard time at 244 shapes of
        2 and 4 ranks, batch 1 - 16, 37 - 2048 tokens per rank, 12 - 32 heads; 0.78 - 1.00 from 5 ms on).  Forward
        only, they pay while the extra launches cost more than the pass, 12 us each at 4 TB/s, or leave CUs idle.  us,
        sequence / per shard:
            W=2 B=8  16 heads D=128 1024 tokens per rank   688 / 657     W=4 B=16 16 heads D=64 (4 kv)  128      132 / 186
            W=2 B=8  16 heads D=64 (4 kv) 1024             254 / 234     W=4 B=4  32 heads D=64         128      129 / 185
            W=2 B=8  12 heads D=64 2048 (idle CUs)         566 / 606     W=2 B=2  16 heads D=64 (4 kv) 2048      185 / 196
        A sequence longer than the backward's q tile lists, or whose rows lie further apart than the kernels' 32-bit tile
        offsets reach, is attended shard by shard."""
        W, B = x.shape[0], x.shape[1]
        attn = self.local_attn
        trained = torch.is_grad_enabled() and (x.requires_grad or any(not isinstance(m, nn.Module) or any(p.requires_grad for p in m.parameters())
                                                                       for m in (attn.wq, attn.wk, attn.wv, attn.wo)))
        if (S_global + 64) * max(self.num_heads, self.num_kv_heads) * self.head_dim >= 0x7fffffff or (trained and S_global > _MAX_BWD_ROWS):
            return False
        if B == 1 or trained:
            return True

        def fill(rows):     # of the CUs, by blocks of 256 rows (under a causal mask a late one and an early one together)
            blocks = B * self.num_heads * -(-rows // 256)
            blocks = -(-blocks // 2) if self.causal and blocks > _CUS else max(blocks, _CUS)
            return blocks / (-(-blocks // _CUS) * _CUS)

        activation = B * S_global * self.num_heads * self.head_dim * x.element_size()
        return 2 * activation < 48e6 * (W - 1) or fill(S_global // W) < fill(S_global)

    def _per_shard(self, x, fc):
        W, B, S_local, _ = x.shape
        H, Hkv, D = self.num_heads, self.num_kv_heads, self.head_dim
        xq = self.local_attn.wq(x).view(W, B, S_local, H, D)
        xk = self.local_attn.wk(x).view(W, B, S_local, Hkv, D)
        xv = self.local_attn.wv(x).view(W, B, S_local, Hkv, D)
        fused = xq.dtype == torch.bfloat16
        table = rope_table(fc, xq.device) if fused else None
        rows = [fc[j * S_local:(j + 1) * S_local] for j in range(W)]
        qs = [xq[j] if fused else rope_one(xq[j], rows[j]) for j in range(W)]
        ks = [rope_one(xk[j], rows[j]) for j in range(W)]       # every K shard once: it is read by every later q shard
        vs, pos, outs = list(xv.unbind(0)), [j * S_local for j in range(W)], []
        for j in range(W):
            n = j + 1 if self.causal else W                     # later shards are fully masked
            outs.append(block_attention(qs[j], ks[:n], vs[:n], pos[:n], pos[j], None, self.causal, q_rope=table)[0])
        return self.local_attn.wo(torch.stack(outs, 0).flatten(3))
