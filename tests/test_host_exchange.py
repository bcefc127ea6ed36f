"""CPU tests of the exchange under tracing: fake GPU tensors have no memory for the compiled copy to read."""
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

import lightron_amd as la
from lightron_amd import parallel_cp as P


def test_exchange_of_fake_gpu_tensors():
    with FakeTensorMode():
        x = torch.empty(2, 3, 8, 4, 16, device="cuda").requires_grad_(True)
        assert P._exchange_node(x) is None
        y = P._all_to_all(x, 2, 1, la.LocalCPGroup(2))
        assert y.shape == (2, 3, 16, 2, 16) and y.device.type == "cuda" and y.grad_fn is not None
        assert P._exchange(y.detach(), 1, 2, 2).shape == x.shape


class _Stub:      # stands for a plain GPU tensor
    is_cuda = True

    def is_conj(self):
        return False

    is_neg = is_conj


def test_tracers_see_the_torch_ops(monkeypatch):
    from lightron_amd import attention
    node = object()
    monkeypatch.setattr(attention, "_cpp_node", lambda: node)
    monkeypatch.setattr(P, "_PLAIN", (_Stub,))
    x = _Stub()
    assert P._exchange_node(x) is node
    with TorchDispatchMode():
        assert P._exchange_node(x) is None
    seen = []
    torch.jit.trace(lambda t: (seen.append(P._exchange_node(x)), t + 1)[1], torch.zeros(2), check_trace=False)
    assert seen and all(s is None for s in seen)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert P._exchange_node(x) is None
