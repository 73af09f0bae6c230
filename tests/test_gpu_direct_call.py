"""Plain eager scans skip the dispatcher; whatever traces, transforms or intercepts a call still
gets the op. Both give the same bits, with and without gradients."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from mamba_amd import selective_scan_hip as ssh
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


def test_functorch_gets_the_op(monkeypatch):
    """torch.func.grad is refused by the op's autograd (a function without setup_context), as when
    the op is called by name; the direct path is not taken."""
    t = {k: v.detach() for k, v in _inputs(False).items()}
    for name in ("_Scan", "_scan_fwd"):  # what a direct call would reach (the op refuses before its kernel)
        monkeypatch.setattr(ssh, name, None)
    f = lambda u: selective_scan_fn(**{**t, "u": u}, delta_softplus=True).sum()
    op = lambda u: torch.ops.mamba_amd.selective_scan_fwd(u, *[t[k] for k in ("delta", "A", "B", "C", "D", "z", "delta_bias")],
                                                          None, None, True, False)[0].sum()
    for call in (f, op):
        with pytest.raises(RuntimeError, match="setup_context"):
            torch.func.grad(call)(t["u"])


def test_conjugate_cotangent_of_the_last_state():
    """A program that conjugates the last state hands back a lazily conjugated gradient, which the
    dispatcher resolves for the op and nothing resolves for a direct call."""
    t = _inputs(True)
    _, last = selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
    w = torch.randn(last.shape, dtype=last.dtype, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    leaves = [v for k, v in t.items() if k != "z"]
    got = torch.autograd.grad((last.conj() * w).real.sum(), leaves, retain_graph=True, allow_unused=True)
    want = torch.autograd.grad(last, leaves, w, allow_unused=True)  # d/dlast of Re(conj(last) w) is w
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert (a - b).abs().max() <= 1e-5 * b.abs().max()


def test_negated_views():
    """The imaginary part of a conjugate is a view whose sign is a flag: read with it, as an input
    (one channel: contiguous at any stride) and as a gradient."""
    t = {k: v.detach()[:, :1].contiguous() if k in ("u", "delta", "z") else v.detach() for k, v in _inputs(False).items()}
    t["A"] = t["A"][:1]
    for k in ("D", "delta_bias"):
        t[k] = torch.complex(t[k][:1], -t[k][:1]).conj().imag
        assert t[k].is_neg() and t[k].is_contiguous()
    plain = {k: v.resolve_neg() for k, v in t.items()}
    leaf = plain["u"].requires_grad_(True)
    t["u"] = leaf
    outs = [selective_scan_fn(**x, delta_softplus=True) for x in (t, plain)]
    assert torch.equal(*outs)
    grads = [torch.autograd.grad(torch.complex(o, o).conj().imag.sum(), leaf)[0] for o in outs]
    assert torch.equal(*grads)


@pytest.mark.parametrize("transform", ["vmap", "forward-mode"])
def test_transforms_meet_the_op(transform):
    """What vmap and forward-mode differentiation make of the op, they make of the public call."""
    t = {k: v.detach() for k, v in _inputs(False).items()}
    op = lambda u: torch.ops.mamba_amd.selective_scan_fwd(u, *[t[k] for k in ("delta", "A", "B", "C", "D", "z", "delta_bias")],
                                                          None, None, True, False)[0]
    fn = lambda u: selective_scan_fn(**{**t, "u": u}, delta_softplus=True)

    def outcome(f):
        try:
            if transform == "vmap":
                return torch.vmap(f)(torch.stack([t["u"], 2 * t["u"]]))
            with torch.autograd.forward_ad.dual_level():
                return torch.autograd.forward_ad.unpack_dual(f(torch.autograd.forward_ad.make_dual(t["u"], t["u"]))).tangent
        except (RuntimeError, NotImplementedError) as e:
            return type(e)

    got, want = outcome(fn), outcome(op)
    assert torch.equal(got, want) if isinstance(want, torch.Tensor) else got is want


def test_a_profiler_sees_the_op():
    t = _inputs(False)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        selective_scan_fn(**t, delta_softplus=True)
    assert any(e.key == "mamba_amd::selective_scan_fwd" for e in prof.key_averages())
