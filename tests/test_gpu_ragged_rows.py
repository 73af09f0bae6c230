"""Rows without 16-byte alignment and rows that end inside a lane's segment: the vector loads
that start before the row's end and are shifted into place, at every remainder of a segment."""
import pytest
import torch

from mamba_amd.selective_scan_hip import selective_scan_fn
from test_conv import run_case as conv_case
from test_gpu_complex import check as check_complex, complex_case
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


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("l", [1, 8, 256, 257, 512, 520, 768, 1024, 1028, 1032, 1536, 2048, 2052])
def test_conv_workgroups_of_fewer_waves(l, dtype):
    """Rows that fill one to four waves of a workgroup, whole vectors or not, and just more."""
    conv_case(2, 5, l, 4, dtype, lens=[l, l // 2], seed=l)


@pytest.mark.parametrize("l,n,lens,io,bc", [
    (l, n, lens, io, bc)
    for l, n, lens in [(8, 4, None), (504, 16, None), (520, 5, [520, 509]), (1032, 3, None), (1024, 16, None), (1028, 4, None),
                       (16, 17, None), (1544, 32, [1537, 700])]
    for io in ("f32", "bf16") for bc in ("f32", "bf16") if n <= 16 or io == bc == "f32"])
def test_rows_of_whole_slots(l, n, lens, io, bc):
    """Rows that are 16-byte multiples but not whole chunks, of one type and of two, and of more than
    16 states: the instances whose lanes clear the slots past the row's end. Also 4-step remainders
    (L = 1028: whole slots in float32 only)."""
    log(f"case whole slots L={l} N={n} {io}/{bc} lens={lens}")
    dtype = "bf16" if "bf16" in (io, bc) else "f32"
    x, dout, dlast = fused_case(3200 + l + n, 2, 13, l, n, dtype, lens=lens)
    td = {"f32": torch.float32, "bf16": torch.bfloat16}
    of = {k: td[bc] if k in "BC" else td[io] for k in ("u", "delta", "z", "B", "C")}
    ts = {k: torch.as_tensor(v).to(dev, of.get(k)) for k, v in x.items()}
    leaves = {k: t.requires_grad_(True) for k, t in ts.items() if k != "seq_lens"}
    out, last = selective_scan_fn(**ts, delta_softplus=True, return_last_state=True)
    d0, d1 = torch.as_tensor(dout).to(dev), torch.as_tensor(dlast).to(dev)
    grads = torch.autograd.grad((out.float() * d0).sum() + (last * d1).sum(), list(leaves.values()))
    for (k, t), g in zip(leaves.items(), grads):
        t.grad = g
    check_fused(ts, out, last, *oracle_fused(x, dout, dlast, False), *tol(dtype))


@pytest.mark.parametrize("l", [8, 508, 520, 1028, 1544])
@pytest.mark.parametrize("dtype,zoh", [("f32", False), ("f32", True), ("bf16", False)])
def test_complex_rows_of_whole_slots(l, dtype, zoh):
    log(f"case complex whole slots L={l} {dtype} zoh={zoh}")
    x, dout, dlast = complex_case(3300 + l, 2, 13, l, 5, dtype, lens=[l, l - 3])
    check_complex(x, dout, dlast, zoh, dtype)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_complex_rows_at_a_misaligned_base(dtype):
    """Complex rows that start one element past an aligned address: the bits of aligned ones (the
    kernels choose by length alone)."""
    log(f"case complex misaligned {dtype}")
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float32
    b, d, l, n = 2, 13, 1544, 5
    g = torch.Generator(device=dev).manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).to(tdt)
    x = dict(u=r(b, d, l), delta=r(b, d, l), z=r(b, d, l), B=r(b, n, l), C=r(b, n, l))
    dout = r(b, d, l)
    A = torch.complex(-torch.exp(r(d, n).float()), 2 * r(d, n).float())

    def moved(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)
        buf[1:].copy_(t.reshape(-1))
        return buf[1:].view(t.shape)

    def run(form):
        ts = {k: form(v).detach().requires_grad_(True) for k, v in x.items()}
        out = selective_scan_fn(ts["u"], ts["delta"], A, ts["B"], ts["C"], z=ts["z"], delta_softplus=True)
        return [out.detach(), *torch.autograd.grad(out, list(ts.values()), form(dout))]

    for i, (a, m) in enumerate(zip(run(torch.clone), run(moved))):
        assert torch.equal(a, m), i
