"""The triangle multiplication's factor and output backwards, each with its products in one pass
(oops_trimul_factor_grads, oops_trimul_output_grads).  The factor pass is held against the separate factor backward (oops_trimul_factors_backward, the same 16-bit projection gradients) and
float64 products of its result: one tile and several runs of tiles, groups that end inside a run, channel and
hidden sizes below 128, with and without a mask and biases."""

import ctypes

import pytest
import torch

from oops_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize(
    "dtype,groups,positions,c,h,masked,biases",
    [
        (torch.bfloat16, 1, 32, 128, 128, True, True),
        (torch.float16, 3, 32 * 5, 128, 128, False, True),
        (torch.bfloat16, 5, 32 * 27, 128, 72, True, False),
        (torch.float16, 2, 32 * 300, 88, 128, True, True),
        (torch.bfloat16, 1, 32 * 2500, 120, 104, True, True),
        (torch.bfloat16, 7, 32 * 310, 128, 128, False, False),
    ],
)
def test_factor_grads(dtype, groups, positions, c, h, masked, biases):
    lib = _lib.load()
    gen = torch.Generator(device=DEV).manual_seed(positions)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    R = groups * positions
    xn = rand(R, c).to(dtype)
    w = (rand(4 * h, c) * c**-0.5).to(dtype)
    bias = rand(4 * h) if biases else None
    mask = (torch.rand(R, device=DEV, generator=gen) > 0.2).float() if masked else None
    gf = rand(2, groups, h, positions).to(dtype)
    before = rand(R, c).to(dtype)
    geo = _lib.TrimulGeometry()
    geo.dtype = _lib.BF16 if dtype == torch.bfloat16 else _lib.F16
    geo.channels, geo.hidden, geo.has_mask = c, h, masked
    geo.groups, geo.positions, geo.c_row, geo.h_row, geo.eps = groups, positions, c, h, 1e-5
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    stream = torch.cuda.current_stream().cuda_stream
    d_proj = torch.empty(4 * h, R, dtype=dtype, device=DEV)
    old_b = torch.empty(lib.oops_trimul_bias_parts(ctypes.byref(geo)), 4 * h, device=DEV)
    assert 0 == lib.oops_trimul_factors_backward(ctypes.byref(geo), ptr(xn), ptr(w), ptr(bias), ptr(mask), ptr(gf),
                                                 ptr(d_proj), None, ptr(old_b), stream), lib.oops_last_error()
    parts = lib.oops_trimul_factor_grad_parts(ctypes.byref(geo))
    assert 1 <= parts <= 256
    d_xn = before.clone()
    wp = torch.full((parts, 4 * h, c), float("nan"), device=DEV)
    bp = torch.full((parts, 4 * h), float("nan"), device=DEV)
    assert 0 == lib.oops_trimul_factor_grads(ctypes.byref(geo), ptr(xn), ptr(w), ptr(bias), ptr(mask), ptr(gf),
                                             ptr(d_xn), ptr(wp), ptr(bp), stream), lib.oops_last_error()
    torch.cuda.synchronize()
    p64, x64, w64 = d_proj.double(), xn.double(), w.double()
    # one rounding of a float32 sum of 4 h + 1 terms: half a unit of the result and the sum's float32 errors
    # (at most 4 h + 1 roundings of 2^-24 of the magnitudes)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    want = before.double() + p64.t() @ w64
    mag = before.double().abs() + p64.t().abs() @ w64.abs()
    assert ((d_xn.double() - want).abs() <= unit * want.abs() + (4 * h + 1) * 2.0**-24 * mag + 1e-7).all()
    # float32 sums over the tokens: at most R roundings of 2^-24 of the magnitudes in any order; the sums here
    # are of runs, so their errors stay far inside sqrt(R) of them
    want, mag = p64 @ x64, p64.abs() @ x64.abs()
    assert ((wp.double().sum(0) - want).abs() <= 4 * R**0.5 * 2.0**-24 * mag + 1e-9).all()
    # the separate backward sums the same float32 values
    want, mag = old_b.double().sum(0), p64.abs().sum(1)
    assert ((bp.double().sum(0) - want).abs() <= 8 * R**0.5 * 2.0**-24 * mag + 1e-6).all()


@pytest.mark.parametrize(
    "dtype,groups,positions,n,c,h,biases",
    [
        (torch.bfloat16, 1, 1, 0, 128, 128, True),  # one row; either side of a 64-row tile
        (torch.float16, 3, 173, 0, 128, 72, False),
        (torch.bfloat16, 1, 64 * 64, 61, 128, 128, True),  # a 61 x 61 pair on a 64 x 64 grid of rows
        (torch.float16, 1, 104 * 104, 99, 96, 128, True),
        (torch.bfloat16, 7, 4097, 0, 120, 104, True),
        (torch.bfloat16, 1, 300 * 300, 0, 128, 128, True),
    ],
)
def test_output_grads(dtype, groups, positions, n, c, h, biases):
    """oops_trimul_output_grads against the separate output backward (oops_trimul_output_backward) and float64
    products of its 16-bit gradients."""

    lib = _lib.load()
    gen = torch.Generator(device=DEV).manual_seed(positions)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=gen)  # noqa: E731
    R = groups * positions
    nrm, xn = rand(R, h).to(dtype), rand(R, c).to(dtype)
    wo, wg = (rand(c, h) * h**-0.5).to(dtype), (rand(c, c) * c**-0.5).to(dtype)
    bo, bg = (rand(c), rand(c)) if biases else (None, None)
    gout = rand(n * n if n else R, c).to(dtype)
    side = round(positions**0.5) if n else 0
    if n:  # the same gradient on the grid of rows
        full = torch.zeros(side, side, c, dtype=dtype, device=DEV)
        full[:n, :n] = gout.view(n, n, c)
        full = full.view(R, c)
    else:
        full = gout
    geo = _lib.TrimulGeometry()
    geo.dtype = _lib.BF16 if dtype == torch.bfloat16 else _lib.F16
    geo.channels, geo.hidden, geo.has_mask = c, h, 0
    geo.groups, geo.positions, geo.c_row, geo.h_row, geo.eps = groups, positions, c, h, 1e-5
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    stream = torch.cuda.current_stream().cuda_stream
    saved = [ptr(t) for t in (nrm, xn, wo, wg, bo, bg)]
    g_val, g_gate = torch.empty(R, c, dtype=dtype, device=DEV), torch.empty(R, c, dtype=dtype, device=DEV)
    assert 0 == lib.oops_trimul_output_backward(ctypes.byref(geo), *saved, ptr(full), ptr(g_val), ptr(g_gate),
                                                stream), lib.oops_last_error()
    parts = lib.oops_trimul_output_grads_parts(ctypes.byref(geo))
    assert 1 <= parts <= 256
    d_nrm, d_xn = torch.empty(R, h, dtype=dtype, device=DEV), torch.empty(R, c, dtype=dtype, device=DEV)
    nan = float("nan")
    wop, wgp = torch.full((parts, c, h), nan, device=DEV), torch.full((parts, c, c), nan, device=DEV)
    bp = torch.full((2, parts, c), nan, device=DEV)
    assert 0 == lib.oops_trimul_output_grads(ctypes.byref(geo), n, side, *saved, ptr(gout), ptr(d_nrm), ptr(d_xn),
                                             ptr(wop), ptr(wgp), ptr(bp), stream), lib.oops_last_error()
    torch.cuda.synchronize()
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for k, (g, w, rows, d, wp) in enumerate(((g_val, wo, nrm, d_nrm, wop), (g_gate, wg, xn, d_xn, wgp))):
        g64, w64, r64 = g.double(), w.double(), rows.double()
        # the gradients themselves may round one way here and the other way there (one unit of each); then one
        # rounding of a float32 sum of c terms
        mag = g64.abs() @ w64.abs()
        flips = unit * mag
        assert ((d.double() - g64 @ w64).abs() <= unit * (g64 @ w64).abs() + flips + c * 2.0**-24 * mag + 1e-7).all()
        mag = g64.abs().t() @ r64.abs()
        bound = 4 * R**0.5 * 2.0**-24 * mag + unit * mag / max(1.0, R**0.5) * 8 + 1e-9
        assert ((wp.double().sum(0) - g64.t() @ r64).abs() <= bound).all()
        # the bias sums take the float32 values: half a unit of each against the rounded ones
        assert ((bp[k].double().sum(0) - g64.sum(0)).abs() <= unit * g64.abs().sum(0) + 1e-6).all()


def test_factor_grads_served_range():
    lib = _lib.load()

    def parts(dtype=_lib.BF16, c=128, h=128, groups=1, positions=64):
        geo = _lib.TrimulGeometry()
        geo.dtype, geo.channels, geo.hidden, geo.has_mask = dtype, c, h, 0
        geo.groups, geo.positions, geo.c_row, geo.h_row, geo.eps = groups, positions, (c + 7) // 8 * 8, (h + 7) // 8 * 8, 1e-5
        return lib.oops_trimul_factor_grad_parts(ctypes.byref(geo))

    assert parts() == 1
    for change in (dict(dtype=_lib.F32), dict(c=64), dict(c=136), dict(c=100), dict(h=64), dict(h=136), dict(positions=81)):
        assert parts(**change) == 0, change


@pytest.mark.parametrize("n,mask_grad", [(32, False), (32, True), (20, False)])
def test_routes_agree(n, mask_grad, monkeypatch):
    """The operator's backward through both passes, through the output pass alone (a mask gradient, or positions
    that are no multiple of 32), and through the separate kernels: every gradient within the roundings of the
    16-bit intermediates that only the separate kernels write (a few units of the largest value)."""

    import oops_amd

    gen = torch.Generator(device=DEV).manual_seed(n)
    rand = lambda *s, scale=1.0: (torch.randn(*s, device=DEV, generator=gen) * scale).bfloat16().requires_grad_()  # noqa: E731
    c = 128
    names = ("input_norm_weight input_norm_bias left_value_weight left_gate_weight right_value_weight "
             "right_gate_weight output_norm_weight output_norm_bias output_weight output_gate_weight").split()
    weights = {k: rand(c) if "norm" in k else rand(c, c, scale=c**-0.5) for k in names}
    biases = {k: rand(c, scale=0.2) for k in ("left_value_bias left_gate_bias right_value_bias right_gate_bias "
                                              "output_bias output_gate_bias").split()}
    pair = rand(n, n, c)
    mask = torch.rand(n, n, device=DEV, generator=gen).requires_grad_(mask_grad)
    dy = rand(n, n, c).detach()
    leaves = [pair, *weights.values(), *biases.values()] + ([mask] if mask_grad else [])

    def grads():
        out = oops_amd.triangle_multiplication(pair, mask, direction="outgoing", **weights, **biases)
        return torch.autograd.grad(out, leaves, dy)

    got = grads()
    lib = _lib.load()
    for name in ("oops_trimul_factor_grad_parts", "oops_trimul_output_grads_parts"):
        monkeypatch.setattr(lib, name, lambda geo: 0)
    for x, y in zip(got, grads()):
        assert (x.double() - y.double()).abs().max() <= 8 * 2.0**-8 * y.double().abs().max()


def test_graph_replays():
    """Both passes under graph capture: every replay equals the eager gradients."""

    import oops_amd

    gen = torch.Generator(device=DEV).manual_seed(5)
    rand = lambda *s: (torch.randn(*s, device=DEV, generator=gen) * 0.3).bfloat16().requires_grad_()  # noqa: E731
    c, n = 128, 48
    names = ("input_norm_weight input_norm_bias left_value_weight left_gate_weight right_value_weight "
             "right_gate_weight output_norm_weight output_norm_bias output_weight output_gate_weight").split()
    weights = {k: rand(c) if "norm" in k else rand(c, c) for k in names}
    pair, dy = rand(n, n, c), rand(n, n, c).detach()
    leaves = [pair, *weights.values()]

    def step():
        return torch.autograd.grad(oops_amd.triangle_multiplication(pair, None, direction="incoming", **weights), leaves, dy)

    want = [g.clone() for g in step()]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        step()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(3):
        for g in got:
            g.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for g, w in zip(got, want))
        step()
        torch.cuda.synchronize()
