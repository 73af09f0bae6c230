"""The reference API's (B, L, D) tensors brought to channel-major rows by one launch."""
import pytest
import torch

from mamba_amd import _lib
from mamba_amd.selective_scan_hip import _to_rows, _transposed, selective_scan

dev = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(1, 1, 1)], [(2, 64, 64), (1, 65, 63)], [(3, 1, 70), (3, 130, 1), (2, 63, 129), (1, 200, 16)],
    [(5, 257, 100), (5, 257, 4)],
])
def test_transposed(shapes):
    print(f"case transposed {shapes}", flush=True)
    xs = [torch.randn(*s, device=dev) for s in shapes]
    for x, y in zip(xs, _transposed(xs)):
        assert y.is_contiguous() and torch.equal(y, x.transpose(1, 2))


@pytest.mark.gpu
def test_layouts_of_the_reference_api():
    """Channel-last, channel-major and strided inputs give the same bits and gradients in their
    own layout's shape."""
    g = torch.Generator(device=dev).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    b, l, d, n = 2, 70, 12, 4
    A, x0, dy = -torch.exp(r(d, n)), r(b, d, n), r(b, l, d)
    base = dict(deltas=r(b, l, d).abs(), Bs=r(b, l, n), Cs=r(b, l, n), u=r(b, l, d))
    forms = {
        "last": lambda v: v.clone(),
        "major": lambda v: v.transpose(1, 2).contiguous().transpose(1, 2),
        "strided": lambda v: torch.stack([v, v], -1)[..., 0],
    }
    assert [x.is_contiguous() for x in _to_rows(*(forms["major"](v) for v in base.values()))] == [True] * 4
    want = None
    for name, form in forms.items():
        t = {k: form(v).requires_grad_(True) for k, v in base.items()}
        y, last = selective_scan(A, initial_x=x0, **t)
        got = [y.detach(), last, *torch.autograd.grad(y, list(t.values()), dy)]
        want = want or got
        for a, w in zip(got, want):
            assert a.shape == w.shape and torch.equal(a, w), name


def test_transpose_validates():
    lib = _lib.register_hip_kernel()
    e = lambda **kw: _lib.TransposeEntry(**{**dict(src=1 << 20, dst=1 << 21, batch=1, rows=8, cols=8), **kw})
    arr = lambda *xs: (_lib.TransposeEntry * len(xs))(*xs)
    bad = _lib.MSS_ERR_INVALID_ARGUMENT
    assert lib.mss_transpose(None, 1, None) == bad
    assert lib.mss_transpose(arr(e()), 0, None) == bad
    assert lib.mss_transpose(arr(*[e()] * 5), 5, None) == bad
    for kw in (dict(src=None), dict(dst=None), dict(batch=0), dict(rows=-1), dict(cols=0), dict(reserved=1),
               dict(dst=(1 << 20) + 128)):
        assert lib.mss_transpose(arr(e(**kw)), 1, None) == bad, kw
    assert lib.mss_transpose(arr(e(), e(src=1 << 22)), 2, None) == bad  # two destinations at one place
    huge = (1 << 31) - 1
    for kw in (dict(batch=huge, rows=huge, cols=huge), dict(rows=huge, cols=huge), dict(batch=huge, rows=1 << 20)):
        assert lib.mss_transpose(arr(e(src=1 << 40, dst=1 << 60, **kw)), 1, None) == _lib.MSS_ERR_UNSUPPORTED, kw
    assert lib.mss_transpose(arr(e(rows=1 << 30, cols=1 << 20, src=1 << 40, dst=1 << 60)), 1, None) == \
        _lib.MSS_ERR_UNSUPPORTED
