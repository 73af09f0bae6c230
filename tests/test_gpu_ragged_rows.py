"""Rows without 16-byte alignment and rows that end inside a lane's segment: the vector loads
that start before the row's end and are shifted into place, at every remainder of a segment."""
import pytest
import torch

from mamba_amd.selective_scan_hip import selective_scan_fn
from test_conv import run_case as conv_case
from test_gpu_parity import check_fused, dev, fused_case, log, oracle_fused, run_fused, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("l", [2, 8, 9, 15, 16, 511, 514, 515, 1021, 1030])
def test_every_segment_remainder(l, dtype):
    log(f"case segment remainder L={l} {dtype}")
    x, dout, dlast = fused_case(3000 + l, 2, 13, l, 5, dtype)
    ts, out, last = run_fused(x, dout, dlast, dtype, False)
    fw, g = oracle_fused(x, dout, dlast, False)
    check_fused(ts, out, last, fw, g, *tol(dtype))


@pytest.mark.parametrize("which", ["io", "bc", "all"])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("l", [1024, 1000])
def test_misaligned_tensors(l, dtype, which):
    """Contiguous tensors that start one element past an aligned address, against the aligned
    ones, forward and backward; also the wide 16-step bf16 forward, whose z rows are copied to
    LDS only when aligned. The same sums in the same order, so the instances may differ by
    float32 contraction only: 1e-6 in the 2-norm, and in bf16 the elements that this moves over
    a rounding boundary (one in 2^8 or so per 2^-24 change, 2^-8 each: far below 1e-4)."""
    log(f"case misaligned L={l} {dtype} {which}")
    b, d = (2, 4096) if dtype == "bf16" else (2, 40)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    g = torch.Generator(device=dev).manual_seed(l)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    x = dict(u=r(b, d, l), delta=r(b, d, l), z=r(b, d, l), B=r(b, 16, l), C=r(b, 16, l))
    x = {k: v.to(tdt) for k, v in x.items()}
    dout = r(b, d, l).to(tdt)
    A, D, bias = -torch.exp(r(d, 16)), r(d), 0.5 * r(d) - 2

    def moved(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)
        buf[1:].copy_(t.reshape(-1))
        return buf[1:].view(t.shape)

    def grads(shift):
        names = {"io": ("u", "delta", "z"), "bc": ("B", "C"), "all": tuple(x)}[which] if shift else ()
        ts = {k: (moved(v) if k in names else v.clone()).requires_grad_(True) for k, v in x.items()}
        out = selective_scan_fn(ts["u"], ts["delta"], A, ts["B"], ts["C"], D=D, z=ts["z"], delta_bias=bias,
                                delta_softplus=True)
        out.backward(moved(dout) if "u" in names else dout)
        return [out] + [t.grad for t in ts.values()]

    for i, (a, m) in enumerate(zip(grads(False), grads(True))):
        assert bool(torch.isfinite(a.float()).all())
        a, m = a.double(), m.double()
        err = float((a - m).norm() / a.norm())
        log(f"  output {i}: {err:.1e}")
        assert err < (1e-6 if dtype == "f32" else 1e-4), i


@pytest.mark.parametrize("layout", ["brl", "rbl"])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("l", [2, 5, 9, 2047, 2050, 4097])
def test_conv_at_any_alignment(l, dtype, layout):
    conv_case(3, 5, l, 4, dtype, layout=layout, lens=[l, l - 1, l // 2], seed=l)
