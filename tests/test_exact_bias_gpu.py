"""Biases whose rows are not 16-byte aligned are added in float32, as the generic kernels add them: finite values
of any size, and the error against float64.  ``rows`` picks the forward's kernel (few rows: the generic one), the
backward's is the fast one unless dO is not aligned; the bias is the same whichever pass runs where."""

import pytest
import torch

from oops_amd import triangle_attention
from oops_amd.attention import _core

from test_triangle_gpu import make_case

pytestmark = pytest.mark.gpu

DEV = "cuda"
NAMES = ("out", "dq", "dk", "dv", "dbias")


def _run(case, shift=False, scale=None):
    q, k, v, mask, bias, dout = case
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v, bias)]
    out = triangle_attention(*leaves[:3], None if mask is None else mask.to(DEV), leaves[3], scale=scale)
    g = dout.to(DEV)
    if shift:  # dO off the 16-byte boundary
        flat = torch.empty(g.numel() + 1, dtype=g.dtype, device=DEV)[1:]
        g = flat.view(g.shape).copy_(g)
        assert g.data_ptr() % 16
    return (out.detach(), *torch.autograd.grad(out, leaves, g))


def _generic(case, scale=None):
    with _core.force_generic():
        return _run(case, scale=scale)


def _finite(tensors):
    for name, t in zip(NAMES, tensors):
        assert bool(t.isfinite().all()), name


@pytest.mark.parametrize("rows,shift", [(3, False), (3, True), (400, False), (400, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_finite_bias_of_any_size(dtype, rows, shift):
    """Query rows whose every key has the lowest finite bias, half of it, two large levels, the largest one."""

    case = make_case(dtype, prefix=(1,), rows=rows, cols=133, head=32, masked=False, seed=3)
    bias, fmin = case[4], torch.finfo(dtype).min
    if dtype == torch.float16:  # (in bfloat16 log2 e times these is infinite: see test_unaligned_bias_gpu.py)
        bias[0, 0, 0, 3] = fmin
        bias[0, 0, 0, 4] = -fmin
        bias[0, 0, 0, 5] = fmin
        bias[0, 0, 0, 5, 40] = -60500.0
        bias[0, 0, 0, 6, ::2] = -65472.0
        bias[0, 0, 0, 6, 1::2] = fmin
    bias[0, 0, 0, 7] = fmin / 2
    bias[0, 0, 0, 8] = -fmin / 2
    bias[0, 0, 0, 9] = fmin / 4
    got, want = _run(case, shift), _generic(case)
    _finite(want)
    _finite(got)
    # (the rows' logits have lost Q.K to float32's rounding of the bias: an equal weight for every key, and P = 1 in
    # the backward, whose LSE has lost the logarithm of their number)
    torch.testing.assert_close(got[0], want[0], rtol=2e-2, atol=2e-2)
    for name, a, b in zip(NAMES[1:], got[1:], want[1:]):
        assert (a - b).float().norm() <= 1e-2 * b.float().norm(), name


@pytest.mark.parametrize("rows,shift", [(3, False), (3, True), (400, False), (400, True)])
@pytest.mark.parametrize("level", [0.3, -0.3, 0.49, -0.49, 0.69, -0.69])
def test_passes_meet_at_large_logits(rows, shift, level):
    """Whole rows at a level of the largest bfloat16: a unit in the last place of such a logit is more than exp2 can
    take, so P = exp2(logit - LSE) needs the forward's and the backward's logits to have the same bits, whichever
    kernels they come from."""

    case = make_case(torch.bfloat16, prefix=(1,), rows=rows, cols=133, head=32, masked=True, seed=12)
    case[4][0, 0, 0, 3:9] = torch.finfo(torch.bfloat16).max * level
    got, want = _run(case, shift), _generic(case)
    _finite(want)
    _finite(got)
    torch.testing.assert_close(got[0], want[0], rtol=2e-2, atol=2e-2)
    for name, a, b in zip(NAMES[1:], got[1:], want[1:]):
        assert (a - b).float().norm() <= 1e-2 * b.float().norm(), name


@pytest.mark.parametrize("rows", [3, 400])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_large_scores_float16(rows, sign):
    """Finite logits beyond the float16 range (64 * 100 * 100 / 8 = 80000) from Q.K alone, 0.8 apart."""

    case = make_case(torch.float16, prefix=(1,), rows=rows, cols=131, head=64, masked=True, seed=4)
    q, k = case[0], case[1]
    q[:, :, :, 0] = 100.0
    k[:, :, :, 0] = sign * 100.0
    k[:, :, :, 0, 0] += torch.arange(131).half() / 16
    got, want = _run(case), _generic(case)
    _finite(want)
    _finite(got)
    # float32 holds such a logit (log2 units) to 2^-7, so P to 0.6%; the passes need not run on the same kernels
    torch.testing.assert_close(got[0], want[0], rtol=2e-2, atol=5e-2)
    for i in (3, 4):  # dV, dBias: dQ and dK multiply that by Q and K
        assert (got[i] - want[i]).float().norm() <= 3e-2 * want[i].float().norm(), NAMES[i]


def _reference(case):
    """Float64 on the CPU."""

    q, k, v, mask, bias, dout = (None if t is None else t.double() if t.is_floating_point() else t for t in case)
    leaves = [t.requires_grad_(True) for t in (q, k, v, bias)]
    qh, kh, vh = (t.transpose(2, 3) for t in leaves[:3])  # (B, R, H, N, D)
    logits = qh @ kh.transpose(-1, -2) * q.shape[-1] ** -0.5 + leaves[3]
    if mask is not None:
        logits = logits.masked_fill(~mask[:, :, None, None, :], float("-inf"))
    out = (torch.softmax(logits, -1).nan_to_num() @ vh).transpose(2, 3)
    return (out.detach(), *torch.autograd.grad(out, leaves, dout))


@pytest.mark.parametrize("dtype,head", [(torch.bfloat16, 32), (torch.bfloat16, 24), (torch.bfloat16, 64),
                                        (torch.float16, 32), (torch.float16, 64)])  # fmt: skip
@pytest.mark.parametrize("spread", [1.0, 60.0])
def test_error_is_the_generic_kernels(dtype, head, spread):
    """The 2-norm errors against float64 are those of the generic kernels (a few percent apart: other tiles, so
    other roundings of P to the dtype), also where Q.K cancels most of a large bias, which an error in the bias's
    weight would show."""

    case = make_case(dtype, prefix=(1,), rows=160, cols=203, head=head, masked=True, seed=11)
    q, k, bias = case[0], case[1], case[4]
    if spread > 1.0:
        b = torch.linspace(-spread, spread, 203)[torch.randperm(203, generator=torch.Generator().manual_seed(1))]
        bias += b.to(dtype)
        q[..., 0] = 1.0
        k[..., 0] = (-b * head**0.5).to(dtype)[None, None, :, None]
    want = _reference(case)
    got, gen = _run(case), _generic(case)
    for name, a, g, w in zip(NAMES, got, gen, want):
        err, ref = ((t.double().cpu() - w).norm() / w.norm() for t in (a, g))
        print(f"{name}: {err:.3e}, generic {ref:.3e}")
        assert err <= 1.05 * ref, f"{name}: {err:.3e}, generic {ref:.3e}"


@pytest.mark.parametrize("scale", [-0.25, 0.0, 1e-6, 1.0, 2.5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_any_scale(dtype, scale):
    case = make_case(dtype, prefix=(1,), rows=200, cols=143, head=40, masked=True, seed=13)
    got, want = _run(case, scale=scale), _generic(case, scale)
    for name, a, b in zip(NAMES, got, want):  # (scale 0: dQ and dK are zeros)
        assert (a - b).float().norm() <= 4 * torch.finfo(dtype).eps * b.float().norm(), name


@pytest.mark.parametrize("rows,shift", [(3, False), (400, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_nonfinite_bias_across_kernels(dtype, rows, shift):
    """A generic forward before a fast backward and the other way round: the same elements are finite, with the
    same values, as with generic kernels alone."""

    case = make_case(dtype, prefix=(1,), rows=rows, cols=133, head=32, masked=True, seed=14)
    bias, inf = case[4], float("inf")
    bias[0, 0, 0, 3, ::2] = -inf
    bias[0, 0, 0, 5] = -inf
    bias[0, 0, 1, 6, 7] = inf
    bias[0, 0, 1, 7, 0] = float("nan")
    got, want = _run(case, shift), _generic(case)
    for name, a, b in zip(NAMES, got, want):
        assert torch.equal(a.isfinite(), b.isfinite()), name
        kept = b.isfinite()
        a, b = a.float()[kept], b.float()[kept]
        assert (a - b).norm() <= 4 * torch.finfo(dtype).eps * b.norm(), name
