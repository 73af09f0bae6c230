"""When a scan may skip the dispatcher: only where nothing traces, transforms or intercepts it and
its tensors are what their memory says."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from mamba_amd import selective_scan_hip as ssh


def test_plain_tensors():
    assert ssh._plain_eager(torch.randn(2), None, torch.nn.Parameter(torch.randn(2)))


def test_intercepted():
    x, seen = torch.randn(3), []
    with TorchDispatchMode():
        assert not ssh._plain_eager(x)
    with torch.autograd.forward_ad.dual_level():
        assert not ssh._plain_eager(x)
    torch.func.grad(lambda v: (seen.append(ssh._plain_eager(x)), v.sum())[1])(x)
    torch.vmap(lambda v: (seen.append(ssh._plain_eager(x)), v)[1])(x)
    assert seen == [False, False]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
        assert not ssh._plain_eager(x)
    assert ssh._plain_eager(x)


def test_other_tensors():
    class Sub(torch.Tensor):
        pass

    assert not ssh._plain_eager(torch.randn(2).as_subclass(Sub))
    conj = torch.randn(2, dtype=torch.complex64).conj()
    assert not ssh._plain_eager(conj.imag)  # a negated view
    for g in (conj, conj.imag, torch._efficientzerotensor((2,))):
        assert not ssh._unflagged(None, g)
    assert ssh._unflagged(torch.randn(2), None)


def test_a_torch_without_these_internals_takes_the_op(monkeypatch):
    monkeypatch.delattr(torch._C, "_len_torch_dispatch_stack")
    monkeypatch.setattr(ssh, "_PROBES", ssh._probes())
    assert not ssh._plain_eager(torch.randn(2))
