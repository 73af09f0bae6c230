"""Scans whose rows are split in time because their channels alone would leave the GPU idle:
every output and gradient against the float64 oracle, at the edges of the split plans."""
import ctypes

import numpy as np
import pytest
import torch

from mamba_amd import _lib
from oracle import scan64
from mamba_amd.selective_scan_hip import selective_scan_fn
from test_gpu_parity import check_fused, close, fused_case, log, oracle_fused, ref_recipe, run_fused, tol
from test_gpu_complex import check as check_complex, complex_case
from test_zz_no_alloc import GRADS, _backward, _forward, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,d,l,n,lens,dtype,zoh", [
    (1, 5, 513, 16, None, "f32", False),       # two chunks, the second of one step
    (8, 192, 2051, 16, None, "f32", False),    # five splits of one chunk, the last of three steps
    (8, 192, 8190, 4, None, "bf16", False),    # sixteen splits of one chunk
    (1, 70, 4096, 11, None, "bf16", True),     # eight splits of one whole chunk, two accumulator copies
    (3, 100, 4100, 16, [4100, 1, 2560], "f32", False),  # rows ending before, at and inside a split
    (3, 100, 4100, 8, [0, 4099, 513], "bf16", True),
])
def test_time_split_scan(b, d, l, n, lens, dtype, zoh):
    log(f"case time split b={b} d={d} l={l} n={n} lens={lens} {dtype} zoh={zoh}")
    x, dout, dlast = fused_case(2000 + l + n, b, d, l, n, dtype, lens=lens, zoh=zoh)
    ts, out, last = run_fused(x, dout, dlast, dtype, zoh)
    fw, g = oracle_fused(x, dout, dlast, zoh)
    check_fused(ts, out, last, fw, g, *tol(dtype))


def bwd_plan(b, d, l, n, lens=None, cplx=False):
    """(splits of a row, chunks of a split, chunks of an adjoint map) of the backward."""
    info = _lib.BwdPlanInfo()
    a = _lib.BwdArgs(batch=b, dim=d, seqlen=l, dstate=n, seq_lens=None if lens is None else 1)
    _lib.check(_lib.register_hip_kernel().mss_bwd_plan_in(a, int(cplx), 1 << 62, info), "mss_bwd_plan_in")
    return info.n_split, info.chunks_per_split, info.chunks_per_map


@pytest.mark.parametrize("b,d,l,n,lens,dtype,zoh,plan", [
    (8, 100, 12003, 2, None, "f32", False, (4, 6, 2)),
    (3, 300, 11003, 3, [11003, 7400, 1300], "bf16", True, (11, 2, 2)),   # rows ending inside a map's chunks
    (8, 100, 12000, 3, [12000, 11000, 4097, 4096, 9000, 6000, 1, 2600], "f32", False, (6, 4, 2)),
    (1, 768, 12000, 1, None, "bf16", False, (4, 6, 2)),
    (2, 400, 12001, 17, None, "f32", False, (4, 6, 2)),                  # two groups of states
])
def test_splits_and_maps_of_several_chunks(b, d, l, n, lens, dtype, zoh, plan):
    log(f"case several chunks b={b} d={d} l={l} n={n} lens={lens} {dtype} zoh={zoh}")
    assert bwd_plan(b, d, l, n, lens) == plan
    x, dout, dlast = fused_case(2000 + l + n, b, d, l, n, dtype, lens=lens, zoh=zoh)
    ts, out, last = run_fused(x, dout, dlast, dtype, zoh)
    check_fused(ts, out, last, *oracle_fused(x, dout, dlast, zoh), *tol(dtype))


@pytest.mark.parametrize("b,d,l,n,lens,zoh,plan", [
    (4, 256, 2051, 3, None, False, (2, 4, 2)),
    (8, 40, 4100, 3, [4100, 4096, 3600, 2561, 1, 2000, 4000, 1025], True, (5, 2, 2)),
])
def test_complex_splits_and_maps_of_several_chunks(b, d, l, n, lens, zoh, plan):
    log(f"case complex several chunks b={b} d={d} l={l} n={n} lens={lens} zoh={zoh}")
    assert bwd_plan(b, d, l, n, lens, cplx=True) == plan
    x, dout, dlast = complex_case(4000 + l + n, b, d, l, n, lens=lens)
    check_complex(x, dout, dlast, zoh)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("how", ["channel-outer", "one element on"])
def test_split_rows_of_other_layouts(cplx, how):
    """Channel-outer rows ([D][B][L]) and rows one element past an aligned address, split in time:
    the bits of contiguous aligned ones (their rows have odd lengths: the same instance of every
    kernel)."""
    log(f"case split layouts cplx={cplx} {how}")
    b, d, l, n = 2, 40, 4099, 4
    assert bwd_plan(b, d, l, n, cplx=cplx)[0] > 1
    g = torch.Generator(device="cuda").manual_seed(8)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = dict(u=r(b, d, l), delta=r(b, d, l), z=r(b, d, l), B=r(b, n, l), C=r(b, n, l))
    dout = r(b, d, l)
    A, D, bias = -torch.exp(r(d, n)), r(d), 0.5 * r(d) - 2
    A = torch.complex(A, 2 * r(d, n)) if cplx else A

    def other(t):
        if how == "channel-outer":
            return t.permute(1, 0, 2).contiguous().permute(1, 0, 2)
        buf = torch.empty(t.numel() + 1, device="cuda")
        buf[1:].copy_(t.reshape(-1))
        return buf[1:].view(t.shape)

    def grads(form):
        ts = {k: form(v).detach().requires_grad_(True) for k, v in x.items()}
        out, last = selective_scan_fn(ts["u"], ts["delta"], A, ts["B"], ts["C"], D=D, z=ts["z"], delta_bias=bias,
                                      delta_softplus=True, return_last_state=True)
        out.backward(form(dout))
        return [out.detach(), last, *[t.grad for t in ts.values()]]

    for i, (a, w) in enumerate(zip(grads(torch.clone), grads(other))):
        assert torch.equal(a, w), i


@pytest.mark.parametrize("n", [16, 20])
def test_backward_in_a_smaller_workspace(n):
    """A workspace that holds the whole-row plan but not the time-split one: the whole-row
    plan runs. Both take the same per-step arithmetic, so the results differ by the order of
    a row's sums only (float32; at most 8 chunks: 1e-5 of the largest value)."""
    lib = _lib.register_hip_kernel()
    b, d, l = 2, 40, 4000
    x, dout, dlast = _inputs(5, b, d, l, n)
    carries, y_pre, out = _forward(lib, x, b, d, l, n)
    full = int(lib.mss_bwd_workspace_bytes(_lib.BwdArgs(batch=b, dim=d, seqlen=l, dstate=n)))
    res = [_backward(lib, lib.mss_bwd, x, carries, y_pre, out, dout, dlast, b, d, l, n,
                     workspace=torch.empty(size, dtype=torch.uint8, device="cuda")) for size in (full, full - 256)]
    for k in GRADS:
        err = (res[0][k] - res[1][k]).abs().max() / res[0][k].abs().max()
        log(f"  {k}: {err:.1e}")
        assert err < 1e-5, k


def test_noalloc_backward_split_in_time():
    """A shape whose time-split plan fits the fixed scratch and whose whole-row plan does not: the
    plan and the bits of mss_bwd in a workspace of the reported size."""
    lib = _lib.register_hip_kernel()
    b, d, l, n = 1, 96, 131072, 16
    log(f"case noalloc split b={b} d={d} l={l} n={n}")
    x, dout, dlast = _inputs(6, b, d, l, n)
    carries, y_pre, out = _forward(lib, x, b, d, l, n)
    size = int(lib.mss_bwd_workspace_bytes(_lib.BwdArgs(batch=b, dim=d, seqlen=l, dstate=n)))
    args = (x, carries, y_pre, out, dout, dlast, b, d, l, n)
    want = _backward(lib, lib.mss_bwd, *args, workspace=torch.empty(size, dtype=torch.uint8, device="cuda"))
    got = _backward(lib, lib.mss_bwd_noalloc, *args)
    for k in GRADS:
        assert bool(torch.isfinite(want[k]).all()) and torch.equal(got[k], want[k]), k


@pytest.mark.parametrize("n", [1, 3, 16])
@pytest.mark.parametrize("grad", [False, True])
def test_state_groups_of_a_forward(n, grad):
    """Four waves to a channel: fewer states than waves, a last round that is not full, steps that
    end inside a wave's share of the outputs; without gradients (no residuals) the same values."""
    from oracle import scan64c
    log(f"case state groups N={n} grad={grad}")
    x, dout, dlast = fused_case(2600 + n, 2, 9, 1290, n, lens=[1290, 515])
    if grad:
        ts, out, last = run_fused(x, dout, dlast, "f32", False)
        check_fused(ts, out, last, *oracle_fused(x, dout, dlast, False))
        return
    with torch.no_grad():
        t = {k: torch.as_tensor(v).cuda() for k, v in x.items()}
        out, last = selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
    fw = scan64c.forward(x["u"], x["delta"], x["A"], x["B"], x["C"], **{k: x[k] for k in x if k not in "uABC" and k != "delta"},
                         delta_softplus=True)
    close("out", out, fw["out"])
    close("last_state", last, fw["last_state"])


def test_forward_workspace():
    """mss_fwd_ws refuses a workspace smaller than its plan's before any launch; mss_fwd, which has
    none, keeps the rows whole and gives the same values up to rounding."""
    lib = _lib.register_hip_kernel()
    b, d, l, n = 1, 64, 4100, 16
    x, _, _ = _inputs(9, b, d, l, n)
    carries, _, out = _forward(lib, x, b, d, l, n)
    split = selective_scan_fn(**x, delta_softplus=True)
    assert (split - out).abs().max() < 1e-5 * out.abs().max()
    p = lambda t: t.data_ptr()
    fa = _lib.FwdArgs(batch=b, dim=d, seqlen=l, dstate=n, u=p(x["u"]), delta=p(x["delta"]), A=p(x["A"]), B=p(x["B"]),
                      C=p(x["C"]), out=p(out))
    need = int(lib.mss_fwd_workspace_bytes(fa))
    assert need > 0
    assert lib.mss_fwd_ws(fa, p(carries), need - 1, None) == _lib.MSS_ERR_WORKSPACE
    assert lib.mss_fwd_ws(fa, None, need, None) == _lib.MSS_ERR_WORKSPACE


@pytest.mark.parametrize("b,d,l,n,lens,dtype,zoh", [
    (1, 40, 4100, 16, None, "f32", False),               # nine chunks, the last of four steps
    (3, 30, 2600, 5, [2600, 1, 1030], "f32", True),      # rows ending before and inside a split
    (2, 50, 3072, 3, None, "bf16", False),               # fewer states than waves of a channel
    (8, 130, 2560, 4, None, "f32", False),               # two splits; several chunks of a channel round
])
def test_complex_time_split(b, d, l, n, lens, dtype, zoh):
    log(f"case complex time split b={b} d={d} l={l} n={n} lens={lens} {dtype} zoh={zoh}")
    x, dout, dlast = complex_case(4000 + l + n, b, d, l, n, dtype, lens=lens)
    check_complex(x, dout, dlast, zoh, dtype)


def test_complex_backward_in_a_smaller_workspace():
    """mss_cbwd runs whole rows in a workspace too small for its time splits (sized without them:
    what the library asked for before a row could be split)."""
    lib = _lib.register_hip_kernel()
    b, d, l, n = 1, 24, 1600, 4
    x, _, _ = complex_case(4100, b, d, l, n, extras=False)
    t = {k: torch.as_tensor(v).cuda() for k, v in x.items()}
    dout = torch.randn(b, d, l, device="cuda")
    out, last, carries, _ = torch.ops.mamba_amd.selective_scan_fwd(t["u"], t["delta"].abs(), t["A"], t["B"], t["C"], None,
                                                                  None, None, None, None, False, False)
    p = lambda v: (torch.view_as_real(v) if v.is_complex() else v).data_ptr()
    res = []
    info = _lib.BwdPlanInfo()
    dims = _lib.BwdArgs(batch=b, dim=d, seqlen=l, dstate=n)
    split_size = int(lib.mss_cbwd_workspace_bytes(dims))
    _lib.check(lib.mss_bwd_plan_in(dims, 1, split_size - 1, info), "mss_bwd_plan_in")
    assert info.n_split == 1
    whole = info.workspace_bytes
    delta = t["delta"].abs()
    for size in (None, whole):
        g = {k: torch.full_like(v, float("nan")) for k, v in dict(u=t["u"], delta=delta, A=t["A"], B=t["B"], C=t["C"]).items()}
        a = _lib.BwdArgs(batch=b, dim=d, seqlen=l, dstate=n, u=p(t["u"]), delta=p(delta), A=p(t["A"]), B=p(t["B"]),
                         C=p(t["C"]), carries=p(carries), dout=p(dout), du=p(g["u"]), ddelta=p(g["delta"]), dA=p(g["A"]),
                         dB=p(g["B"]), dC=p(g["C"]))
        need = int(lib.mss_cbwd_workspace_bytes(a))
        assert need > whole
        ws = torch.empty(size or need, dtype=torch.uint8, device="cuda")
        a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
        _lib.check(lib.mss_cbwd(a, None), "mss_cbwd")
        torch.cuda.synchronize()
        res.append(g)
    for k in res[0]:
        x0, x1 = (torch.view_as_real(r[k]) if r[k].is_complex() else r[k] for r in res)
        assert bool(torch.isfinite(x0).all())
        assert (x0 - x1).abs().max() < 1e-5 * x0.abs().max(), k


@pytest.mark.parametrize("b,d,l,n", [(1, 256, 8192, 16), (2, 96, 4100, 20)])
def test_reference_backward_split_in_time(b, d, l, n):
    """mss_scan_bwd and mss_scan_bwd_ws at shapes whose time-split plan needs less workspace than
    the whole-row one (the second: over two groups of states), in the size the library reports."""
    log(f"case reference backward b={b} d={d} l={l} n={n}")
    lib = _lib.register_hip_kernel()
    A, deltas, Bs, Cs, u, x0 = ref_recipe(15, batch=b, length=l, dim=d, n=n)
    rng = np.random.default_rng(16)
    dy, dfin = rng.standard_normal((b, l, d)).astype(np.float32), rng.standard_normal((b, d, n)).astype(np.float32)
    T = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
    tr = lambda a: T(np.swapaxes(a, 1, 2))
    ins = [T(A), tr(deltas), tr(Bs), tr(Cs), tr(u), T(x0)]
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    y, fin = torch.empty(b, d, l, device="cuda"), torch.empty(b, d, n, device="cuda")
    cs = torch.empty(b, d, -(-l // 2048), n, 2, device="cuda")
    _lib.check(lib.mss_scan_fwd(None, 0, b, l, d, n, *map(P, ins), P(y), P(fin), P(cs)), "mss_scan_fwd")
    cot = [tr(dy), T(dfin)]
    res = []
    for ws in (None, torch.empty(int(lib.mss_scan_bwd_workspace_bytes(b, l, d, n)), dtype=torch.uint8, device="cuda")):
        outs = [torch.full_like(t, float("nan")) for t in ins]
        args = (None, b, l, d, n, *map(P, ins), P(cs), *map(P, cot), *map(P, outs))
        _lib.check(lib.mss_scan_bwd(*args) if ws is None else lib.mss_scan_bwd_ws(*args, P(ws), ws.numel()), "mss_scan_bwd")
        torch.cuda.synchronize()
        res.append(outs)
    grads, ab = scan64.reference_api_backward(A, deltas, Bs, Cs, u, x0, dy, dfin, abs_terms=True)
    for name, o, w, g in zip(["dA", "ddeltas", "dBs", "dCs", "du", "dinitial_x"], *res, grads):
        assert torch.equal(o, w), name
        close(name, o if o.shape == g.shape else o.transpose(1, 2), g, scale=ab.get(name))


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("backward", [False, True])
def test_growth_over_a_split_from_nothing(cplx, backward):
    """A growing state (Re A > 0) that is zero, and an adjoint that is zero, stay zero over a split
    or map whose product of a_bar overflows float32 (e^120; a chunk's e^60 does not): the outputs of
    the same call with those steps' delta zero."""
    b, d, l, n = ((8, 40, 4100, 3) if cplx else (1, 768, 12000, 1)) if backward else ((1, 160, 8192, 2) if cplx else (1, 500, 4096, 4))
    if backward:
        assert bwd_plan(b, d, l, n, cplx=cplx)[2] == 2
        still = slice(3072, 4096) if cplx else slice(10240, 11264)  # the two chunks of a map
    else:
        lib = _lib.register_hip_kernel()
        a = _lib.FwdArgs(batch=b, dim=d, seqlen=l, dstate=n)
        per = (2, 4) if cplx else (3, 2)  # chunks of a split, floats of a map
        need = (lib.mss_cfwd_workspace_bytes if cplx else lib.mss_fwd_workspace_bytes)(a)
        assert need == (-(-(l // 512) // per[0]) - 1) * b * d * n * per[1] * 4
        still = slice(0, per[0] * 512)
    log(f"case growth cplx={cplx} backward={backward}")
    g = torch.Generator(device="cuda").manual_seed(21)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    u, delta, B, C, dout = r(b, d, l), 1e-3 * r(b, d, l).abs(), r(b, n, l), r(b, n, l), r(b, d, l)
    A = torch.full((d, n), 60 / 512, device="cuda")
    A = torch.complex(A, r(d, n)) if cplx else A
    if backward:
        u.zero_()
        dout[..., still.start:] = 0
    else:
        u[..., still] = 0
    res = []
    for step in (0.0, 1.0):
        delta[..., still] = step
        leaves = [t.clone().requires_grad_(backward) for t in (u, delta, A, B, C)]
        out, last = selective_scan_fn(*leaves, return_last_state=True)
        res.append([out, last, *(torch.autograd.grad(out, leaves, dout) if backward else ())])
    for i, (want, got) in enumerate(zip(*res)):
        want, got = (torch.view_as_real(t.detach()) if t.is_complex() else t.detach() for t in (want, got))
        assert bool(torch.isfinite(want).all()) and torch.equal(got, want), i


@pytest.mark.parametrize("b,d,l,n,dtype,zoh,cplx", [
    (1, 300, 700, 1, "f32", False, False), (1, 300, 700, 2, "f32", False, False),   # a workgroup a CU or fewer
    (1, 600, 700, 7, "f32", False, False), (1, 600, 700, 8, "f32", False, False),   # two
    (1, 600, 700, 3, "bf16", False, False), (1, 600, 700, 4, "bf16", False, False),
    (1, 1100, 700, 6, "f32", True, False), (1, 1100, 700, 7, "f32", True, False),   # three
    (1, 1100, 700, 11, "bf16", False, False), (1, 1100, 700, 12, "bf16", False, False),
    (1, 300, 700, 2, "f32", False, True), (1, 300, 700, 3, "f32", False, True),     # two waves a SIMD or fewer
    (1, 600, 700, 3, "f32", False, True), (1, 600, 700, 3, "f32", True, True), (1, 200, 700, 2, "f32", False, True),
])
def test_states_at_which_waves_share_a_channel(b, d, l, n, dtype, zoh, cplx):
    """Either side of the state counts from which four waves share a channel."""
    log(f"case sharing b={b} d={d} l={l} n={n} {dtype} zoh={zoh} cplx={cplx}")
    if cplx:
        x, dout, dlast = complex_case(4200 + d + n, b, d, l, n, dtype)
        check_complex(x, dout, dlast, zoh, dtype)
        return
    x, dout, dlast = fused_case(4200 + d + n, b, d, l, n, dtype, zoh=zoh)
    ts, out, last = run_fused(x, dout, dlast, dtype, zoh)
    check_fused(ts, out, last, *oracle_fused(x, dout, dlast, zoh), *tol(dtype))
