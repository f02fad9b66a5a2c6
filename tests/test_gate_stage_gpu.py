"""The gated output stage as one pass over its rows (oops_gate_stage_*, oops_linear_grad_products): values and
gradients against the same formula in float64 on the same 16-bit inputs, at the edges of its row tiles (32 and
64), of its 128-column blocks and of its 256- and 384-channel ranges, over strided operands, with infinite
inputs, and the forms it hands to the separate operators (missing gradients, a second derivative)."""

import pytest
import torch

import oops_amd
from oops_amd.attention import gate as G

pytestmark = pytest.mark.gpu

UNIT = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _inputs(dtype, prefix, heads, q, d, c, o, layout="qhd", seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    n = heads * d
    if layout == "hqd":  # head-major in memory
        att = rand(*prefix, heads, q, d).to(dtype)
    else:  # token-major in memory, read through its strides
        att = rand(*prefix, q, heads, d).to(dtype).transpose(-3, -2)
    single = rand(*prefix, q, c).to(dtype)
    if layout == "wide":  # rows and weights inside wider buffers
        single = torch.cat([single, single], -1)[..., :c]
    wg = (rand(n, c) * c**-0.5).to(dtype)
    wo = (rand(o, n) * n**-0.5).to(dtype)
    if layout == "wide":
        wg, wo = torch.cat([wg, wg], 1)[:, :c], torch.cat([wo, wo], 1)[:, :n]
    return [t.detach().requires_grad_() for t in (att, single, wg, wo)]


def _reference(att, single, wg, wo, grad):
    """Float64 values, gradients, and for each the sum of the magnitudes of its terms."""

    a, s, g, w = (t.detach().double().requires_grad_() for t in (att, single, wg, wo))
    rows = a.transpose(-3, -2).flatten(-2)
    gate = torch.sigmoid(s @ g.t())
    out = (gate * rows) @ w.t()
    grads = torch.autograd.grad(out, (a, s, g, w), grad.double())
    with torch.no_grad():
        # magnitudes: |operand| sums through the same chain (|sigmoid'| <= gate (1 - gate))
        mrows, mgrad = rows.abs(), grad.double().abs()
        m_out = (gate * mrows) @ w.abs().t()
        m_gated = mgrad @ w.abs()
        m_att = (m_gated * gate).unflatten(-1, (a.shape[-3], a.shape[-1])).transpose(-3, -2)
        m_logit = m_gated * mrows * gate * (1 - gate)
        # an error of the logits (their magnitude sum) moves every later value through the sigmoid's slope
        m_lin = s.abs() @ g.abs().t()
        m_out = m_out + (gate * (1 - gate) * m_lin * mrows) @ w.abs().t()
        m_att = m_att + (m_gated * gate * (1 - gate) * m_lin).unflatten(
            -1, (a.shape[-3], a.shape[-1])).transpose(-3, -2)
        m_logit = m_logit * (1 + m_lin) + m_gated * mrows * (1 - gate) * 1.0
        m_single = m_logit @ g.abs()
        m_wg = m_logit.flatten(0, -2).t() @ s.abs().flatten(0, -2)
        m_wo = mgrad.flatten(0, -2).t() @ (gate * mrows * (1 + m_lin)).flatten(0, -2)
    return (out, *grads), (m_out, m_att, m_single, m_wg, m_wo)


def _check(dtype, got, want, magnitude):
    """Every value is a sum of products whose factors carry at most eight roundings to the 16-bit type (logits,
    gate, gated / grad_gated, the three steps of the sigmoid's backward, the products' result), each of half a
    unit: |error| <= 8 * unit / 2 * (sum of the terms' magnitudes), plus float32 sums (negligible against it)."""

    for name, x, y, m in zip(("out", "attention", "single", "gate_weight", "output_weight"), got, want, magnitude):
        assert x.dtype == dtype
        excess = ((x.double() - y).abs() - 4 * UNIT[dtype] * m - 1e-6).max().item()
        assert excess <= 0, (name, excess)


CASES = [
    # prefix, heads, q, d, c, o: one row, either side of the row tiles and of the column blocks, full width
    ((1,), 1, 1, 16, 8, 8),
    ((1,), 2, 31, 16, 40, 24),
    ((2,), 4, 33, 32, 128, 128),
    ((3, 5), 8, 13, 16, 128, 64),
    ((1,), 8, 65, 32, 256, 256),
    ((2,), 9, 127, 16, 136, 120),
    ((1,), 4, 129, 64, 256, 8),
    ((3,), 5, 45, 24, 96, 40),  # 120 channels in 16-channel runs
    ((3,), 17, 45, 8, 96, 136),
    ((1,), 16, 200, 16, 72, 256),
    ((1,), 16, 95, 24, 384, 384),  # the wide forward: more than 256 channels somewhere
    ((2,), 11, 33, 24, 16, 40),
    ((1,), 2, 129, 16, 264, 8),
    ((3,), 4, 31, 32, 72, 376),
    ((2, 9), 4, 997, 32, 64, 128),
    ((5,), 8, 4001, 32, 256, 256),
]


@pytest.mark.parametrize("layout", ["hqd", "qhd", "wide"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, (*c[0], *c[1:]))))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_stage(dtype, case, layout):
    prefix, heads, q, d, c, o = case
    att, single, wg, wo = _inputs(dtype, prefix, heads, q, d, c, o, layout)
    att5, rows, weight = G._operands(att.transpose(-3, -2), single, wg, dtype)
    assert G._stage_ok(att5, rows, weight, wo)
    out = oops_amd.gate_attention_output(att, single, wg, wo)
    grad = torch.randn(out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(1)).to(dtype)
    grads = torch.autograd.grad(out, (att, single, wg, wo), grad)
    want, magnitude = _reference(att, single, wg, wo, grad)
    _check(dtype, (out, *grads), want, magnitude)
    with torch.no_grad():  # the form that keeps no logits: the same values
        assert torch.equal(oops_amd.gate_attention_output(att, single, wg, wo), out)


def test_gate_stage_matches_the_separate_operators():
    """The same roundings: attention and logit gradients bit for bit, up to the float32 order of the products."""

    att, single, wg, wo = _inputs(torch.bfloat16, (4,), 8, 300, 32, 256, 256)
    att5, rows, weight = G._operands(att.transpose(-3, -2), single, wg, torch.bfloat16)
    out, logits = G._stage_forward(att5, rows, weight, wo, True)
    gated, want_logits = G._forward_impl(att5, rows, weight, True)
    assert torch.equal(logits, want_logits)
    torch.testing.assert_close(out, torch.nn.functional.linear(gated, wo), rtol=2**-7, atol=1e-3)


def test_gate_stage_missing_gradients_and_second_derivative():
    dtype = torch.bfloat16
    full = _inputs(dtype, (2,), 4, 70, 32, 128, 128)
    grad = torch.ones(2, 70, 128, device="cuda", dtype=dtype)
    want, magnitude = _reference(*full, grad)
    for wanted in ((0,), (3,), (1, 2), (0, 3), (1, 3), (0, 1, 3), (0, 2, 3)):
        operands = [t.detach().requires_grad_(i in wanted) for i, t in enumerate(full)]
        out = oops_amd.gate_attention_output(*operands)
        grads = torch.autograd.grad(out, [operands[i] for i in wanted], grad)
        _check(dtype, grads, [want[1 + i] for i in wanted], [magnitude[1 + i] for i in wanted])
    # under create_graph: first derivatives with derivatives of their own, and no mixing of operands that
    # depend on each other
    att, single, wg, wo = full
    dependent = att + single.sum() * 0.25
    out = oops_amd.gate_attention_output(dependent, single, wg, wo)
    (g_first,) = torch.autograd.grad(out, (dependent,), grad, create_graph=True, retain_graph=True)
    (second,) = torch.autograd.grad(g_first.float().square().sum(), (wo,))
    assert second.shape == wo.shape and second.abs().max() > 0
    (got,) = torch.autograd.grad(out, (single,), grad, create_graph=True, retain_graph=True)
    (plain,) = torch.autograd.grad(out, (single,), grad)
    torch.testing.assert_close(got, plain, rtol=2**-6, atol=0.02 * plain.abs().max().item())


def test_gate_stage_not_served():
    """Operands outside the one-pass kernels' range keep the separate operators."""

    served = dict(dtype=torch.bfloat16, prefix=(1,), heads=4, q=9, d=32, c=128, o=128)
    for change in (dict(dtype=torch.float32), dict(d=20), dict(c=392), dict(o=392), dict(heads=13), dict(o=12), dict(c=12),
                   dict(c=384, q=16385)):  # fmt: skip
        att, single, wg, wo = _inputs(**{**served, **change})
        att5, rows, weight = G._operands(att.transpose(-3, -2), single, wg, att.dtype)
        assert not G._stage_ok(att5, rows, weight, wo)
        out = oops_amd.gate_attention_output(att, single, wg, wo)
        assert out.shape == (*single.shape[:-1], wo.shape[0])


@pytest.mark.parametrize("heads,c,o", [(5, 128, 128), (9, 64, 136), (11, 72, 264)])
def test_gate_stage_infinite_inputs(heads, c, o):
    """An infinite input saturates the gates of its row; channels that only pad the kernels' tiles add nothing."""

    att, single, wg, wo = (t.detach() for t in _inputs(torch.bfloat16, (1,), heads, 40, 24, c, o))
    single[0, 3, 5] = float("inf")
    att[0, 1, 7, 2] = float("-inf")
    att5, rows, weight = G._operands(att.transpose(-3, -2), single, wg, torch.bfloat16)
    assert G._stage_ok(att5, rows, weight, wo)
    gate = torch.sigmoid((single.double() @ wg.double().t()).float())
    want = (gate.bfloat16() * att.transpose(-3, -2).flatten(-2)).double() @ wo.double().t()
    got = oops_amd.gate_attention_output(att, single, wg, wo)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert got[0, 3].isfinite().all()


@pytest.mark.parametrize("c", [256, 384])
def test_gate_stage_graph_replays(c):
    operands = _inputs(torch.bfloat16, (2,), c // 32, 150, 32, c, c)
    grad = torch.randn(2, 150, c, device="cuda").bfloat16()

    def step():
        return torch.autograd.grad(oops_amd.gate_attention_output(*operands), operands, grad)

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


@pytest.mark.parametrize("c", [128, 384])
def test_tangent_of_output_weight(c):
    """The output is linear in the output weight, so its tangent is the stage of the weight's; with gradients the
    projection refuses forward mode."""

    att, single, wg, wo = _inputs(torch.bfloat16, (1,), 4, 40, 32, c, c)
    tangent = torch.randn_like(wo)
    with torch.autograd.forward_ad.dual_level():
        with torch.no_grad():
            dual = torch.autograd.forward_ad.make_dual(wo.detach(), tangent)
            out = torch.autograd.forward_ad.unpack_dual(oops_amd.gate_attention_output(att, single, wg, dual))
            want = oops_amd.gate_attention_output(att, single, wg, tangent)
        assert out.tangent is not None
        torch.testing.assert_close(out.tangent, want, rtol=2.0**-6, atol=2.0**-6)
        with pytest.raises(RuntimeError):
            oops_amd.gate_attention_output(att, single, wg, torch.autograd.forward_ad.make_dual(wo, tangent))


@pytest.mark.parametrize("dtype,c", [(torch.bfloat16, 64), (torch.bfloat16, 512), (torch.float32, 64)])
def test_lazily_negated_operands(dtype, c):
    """Negated views of each operand and of the gradient, in one pass (64 channels) and in separate operators."""

    leaves = _inputs(dtype, (2,), 2, 33, c // 2, c, c)
    grad = torch.randn(2, 33, c, device="cuda").to(dtype)

    def run(operands, g):
        out = oops_amd.gate_attention_output(*operands)
        return (out, *torch.autograd.grad(out, leaves, g))

    want = run(leaves, grad)
    for i in range(5):
        neg = [torch._neg_view(-t) if i == j else t for j, t in enumerate(leaves)]
        g = torch._neg_view(-grad) if i == 4 else grad
        assert (neg + [g])[i].is_neg()
        for a, b in zip(run(neg, g), want):
            torch.testing.assert_close(a, b)


class _Wrapped(torch.Tensor):
    """A wrapper without storage of its own, as quantised and distributed tensors are."""

    @staticmethod
    def __new__(cls, inner):
        out = torch.Tensor._make_wrapper_subclass(cls, inner.shape, strides=inner.stride(), dtype=inner.dtype,
                                                  device=inner.device)  # fmt: skip
        out.inner = inner
        return out

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        unwrap = lambda t: t.inner if isinstance(t, cls) else t  # noqa: E731
        return func(*torch.utils._pytree.tree_map(unwrap, args), **(kwargs or {}))


@pytest.mark.parametrize("which", [1, 2, 3])
@pytest.mark.parametrize("c", [128, 512])
def test_subclass_operands(which, c):
    """A wrapper in the place of single, gate weight or output weight is dispatched, not read."""

    operands = [t.detach() for t in _inputs(torch.bfloat16, (1,), 4, 48, c // 4, c, c)]
    want = oops_amd.gate_attention_output(*operands)
    operands[which] = _Wrapped(operands[which])
    with torch.no_grad():
        got = oops_amd.gate_attention_output(*operands)
    got = got.inner if isinstance(got, _Wrapped) else got
    torch.testing.assert_close(got, want, rtol=2.0**-6, atol=2.0**-6)


def test_far_apart_rows():
    """Rows of `single` 4M elements apart: the forward takes them, so the backward does."""

    dtype, c, rows = torch.bfloat16, 64, 5
    att, _, wg, wo = _inputs(dtype, (1,), 2, rows, c // 2, c, c)
    single = torch.randn(1, rows, 1 << 22, device="cuda", dtype=dtype)[..., :c].requires_grad_()
    grad = torch.randn(1, rows, c, device="cuda").to(dtype)

    def run(s):
        out = oops_amd.gate_attention_output(att, s, wg, wo)
        return (out, *torch.autograd.grad(out, (att, s, wg, wo), grad))

    for a, b in zip(run(single), run(single.detach().contiguous().requires_grad_())):
        assert torch.equal(a, b)


@pytest.mark.parametrize("c", [136, 256])
def test_rows_around_the_streaming_forward(c):
    """The last row count of the streaming forward and the first of the one that keeps its weights: the same sums
    in the same order, so the same bits."""

    att, single, wg, wo = (t.detach() for t in _inputs(torch.bfloat16, (1,), c // 8, 8193, 8, c, c))
    more = oops_amd.gate_attention_output(att, single, wg, wo)
    fewer = oops_amd.gate_attention_output(att[:, :, :8192], single[:, :8192], wg, wo)
    assert torch.equal(more[:, :8192], fewer)


@pytest.mark.parametrize("rows", [48, 300])
def test_captured_training_step(rows):
    """Replays on new inputs, with eager work between them: the bits of eager calls."""

    static = _inputs(torch.bfloat16, (1,), 16, rows, 24, 384, 384)
    grad = torch.randn(1, rows, 384, device="cuda").to(torch.bfloat16)

    def step(x):
        out = oops_amd.gate_attention_output(*x)
        return (out, *torch.autograd.grad(out, x, grad))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step(static)
    for seed in range(1, 4):
        fresh = _inputs(torch.bfloat16, (1,), 16, rows, 24, 384, 384, seed=seed)
        with torch.no_grad():
            for a, b in zip(static, fresh):
                a.copy_(b)
        graph.replay()
        got = [t.clone() for t in captured]
        for a, b in zip(got, step(fresh)):
            assert torch.equal(a, b)
