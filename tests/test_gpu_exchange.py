"""The Ulysses exchange on the GPU (ltr_copy_strided behind SeqAllToAll): bit-exact against the oracle's split / all_to_all / cat."""
import pytest
import torch

from oracle import ring_attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,shape,scatter,gather,dtype", [
    (4, (2, 5, 8, 64), 2, 1, torch.bfloat16),       # sequence -> heads, runs of two heads
    (4, (2, 20, 2, 64), 1, 2, torch.bfloat16),      # and back
    (2, (1, 7, 6, 24), 2, 1, torch.float32),        # odd lengths: runs of 288 bytes
    (3, (3, 4, 3, 8), 2, 1, torch.bfloat16),        # one 16-byte vector per run
    (2, (2, 3, 4, 6), 2, 1, torch.bfloat16),        # 24-byte runs: not the kernel's
    (2, (5, 4, 6), -1, 0, torch.float32),           # negative dims, a scattered last dim
    (2, (4, 130, 32, 128), 2, 1, torch.bfloat16),   # more than one block, a ragged last one
])
def test_exchange_matches_the_oracle(ltr, W, shape, scatter, gather, dtype):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(W, *shape, generator=g).to(dtype)
    grp = ltr.LocalCPGroup(W)
    xd = x.cuda().requires_grad_(True)
    nd = len(shape)
    want = orc.seq_all_to_all([x[r] for r in range(W)], scatter % nd, gather % nd)
    for y in (ltr._all_to_all(xd, scatter, gather, grp), ltr.SeqAllToAll.apply(xd, scatter, gather, grp)):
        assert y.is_contiguous() and all(torch.equal(y[r].cpu(), want[r]) for r in range(W))
        gy = torch.randn(y.shape, generator=g).to(dtype)
        xd.grad = None
        y.backward(gy.cuda())
        back = orc.seq_all_to_all([gy[r] for r in range(W)], gather % nd, scatter % nd)
        assert all(torch.equal(xd.grad[r].cpu(), back[r]) for r in range(W))
    # views: heads in front of the sequence, and a slice that starts off a 16-byte boundary
    if len(shape) == 4:
        xt = x.transpose(2, 3).contiguous().cuda().transpose(2, 3)
        assert torch.equal(ltr._all_to_all(xt, scatter, gather, grp).cpu(), torch.stack(want))
        xo = torch.empty(x.numel() + 1, dtype=dtype, device="cuda")[1:].view(x.shape)
        xo.copy_(x)
        assert torch.equal(ltr._all_to_all(xo, scatter, gather, grp).cpu(), torch.stack(want))


def test_gradients_may_be_conjugated_views(ltr):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(2, 3, 4, 8, generator=g, dtype=torch.complex64).cuda().requires_grad_(True)
    gy = torch.randn(2, 3, 8, 4, generator=g, dtype=torch.complex64)
    ltr._all_to_all(x, 2, 1, ltr.LocalCPGroup(2)).backward(gy.cuda().conj())
    want = torch.stack(orc.seq_all_to_all(list(gy.conj().resolve_conj()), 1, 2))
    assert torch.equal(x.grad.cpu(), want)
