"""Plain eager scans skip the dispatcher; whatever traces, transforms or intercepts a call still
gets the op. Both give the same bits, with and without gradients."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from mamba_amd.selective_scan_hip import selective_scan_fn

pytestmark = pytest.mark.gpu


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def _inputs(cplx):
    g = torch.Generator().manual_seed(11 + cplx)
    r = lambda *s: torch.randn(*s, generator=g)
    b, d, l, n = 2, 6, 300, 4
    A = -torch.exp(r(d, n))
    A = torch.complex(A, 2 * r(d, n)) if cplx else A
    t = dict(u=r(b, d, l), delta=r(b, d, l), A=A, B=r(b, n, l), C=r(b, n, l), D=r(d), z=r(b, d, l), delta_bias=r(d))
    return {k: v.cuda().requires_grad_(True) for k, v in t.items()}


def _step(t, use_last):
    out, last = selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
    loss = out.square().sum()
    if use_last:
        loss = loss + (torch.view_as_real(last) if last.is_complex() else last).square().sum()
    return [out.detach(), last.detach(), *torch.autograd.grad(loss, list(t.values()))]


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("use_last", [False, True])
def test_direct_and_op_paths_agree(cplx, use_last):
    t = _inputs(cplx)
    direct = _step(t, use_last)
    with Seen() as seen:
        op = _step(t, use_last)
    assert any("selective_scan_fwd" in n for n in seen.names)
    for a, b in zip(direct, op):
        assert torch.equal(a, b)
    with torch.no_grad():
        out, last = selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
    assert torch.equal(out, direct[0]) and torch.equal(last, direct[1])


def test_only_the_last_state_differentiated():
    t = _inputs(False)
    _, last = selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
    g = torch.autograd.grad(last.sum(), [t["u"], t["C"]], allow_unused=True)
    assert bool(torch.isfinite(g[0]).all()) and g[0].abs().max() > 0
    assert g[1] is None or not g[1].any()


def test_second_differentiation_is_refused():
    t = _inputs(False)
    out = selective_scan_fn(**t, delta_softplus=True)
    (gu,) = torch.autograd.grad(out.sum(), [t["u"]], create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(gu.sum(), [t["delta"]])


def test_saved_tensor_hooks_see_the_residuals():
    t = _inputs(False)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(x.shape) or x, lambda x: x):
        out = selective_scan_fn(**t, delta_softplus=True)
    assert torch.Size((2, 6, 4, 38)) in packed  # the carries: one state per 8 steps
    out.sum().backward()
    assert t["u"].grad is not None


def test_functorch_gets_the_op():
    t = {k: v.detach() for k, v in _inputs(False).items()}
    f = lambda u: selective_scan_fn(**{**t, "u": u}, delta_softplus=True).sum()
    u = t["u"].clone().requires_grad_(True)
    (want,) = torch.autograd.grad(f(u), [u])
    try:
        got = torch.func.grad(f)(t["u"])
    except RuntimeError:
        return  # refused by the op, as before
    assert torch.equal(got, want)
