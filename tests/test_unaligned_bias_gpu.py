"""Shared biases whose rows are not 16-byte aligned (key counts that are no multiple of 8) on the 16-bit
fast kernels: against the oracle at the edges of the 32- and 64-key tiles and of the fused backward's
geometries, and against the generic kernels where the bias is not finite.  The tolerance is that of the
other 16-bit cases (accuracy.py)."""

import pytest
import torch

from oops_amd import pair_bias_attention, triangle_attention
from oops_amd.attention import _core

from accuracy import assert_close
from oracle import attention as ora
from test_triangle_gpu import _np, make_case, run_and_check

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cols,head,rows", [(1, 32, 2), (31, 32, 3), (33, 16, 900), (65, 32, 3), (95, 24, 600), (129, 32, 300),
                                            (257, 64, 3), (289, 64, 2), (387, 32, 2), (387, 48, 2), (771, 32, 2),
                                            (1027, 32, 1)])  # fmt: skip
def test_against_oracle(dtype, cols, head, rows):
    case = make_case(dtype, prefix=(1,), rows=rows, cols=cols, head=head, masked=cols % 4 == 3, seed=cols,
                     layout="swapped" if cols % 3 == 0 else "dense")  # fmt: skip
    run_and_check(*case, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bias_view_rows(dtype):
    """An aligned row length at a misaligned offset, rectangular queries, two batch elements."""

    g = torch.Generator().manual_seed(5)
    q = torch.randn(2, 3, 2, 45, 32, generator=g).to(dtype)
    k, v = (torch.randn(2, 3, 2, 72, 32, generator=g).to(dtype) for _ in range(2))
    wide = torch.randn(2, 1, 2, 45, 80, generator=g).to(dtype)
    dout = torch.randn(2, 3, 2, 45, 32, generator=g).to(dtype)
    lq, lk, lv = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    bias = wide.to(DEV)[..., 3:75].requires_grad_(True)
    out = pair_bias_attention(lq, lk, lv, None, bias)
    grads = torch.autograd.grad(out, (lq, lk, lv, bias), dout.to(DEV))
    with _core.force_generic():
        want = pair_bias_attention(lq, lk, lv, None, bias)
        wants = torch.autograd.grad(want, (lq, lk, lv, bias), dout.to(DEV))
    for got, ref, name in zip((out, *grads), (want, *wants), ("out", "dq", "dk", "dv", "dbias")):
        assert_close(got, _np(ref), dtype, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
def test_nonfinite_bias_as_generic(dtype, masked):
    """(400 rows: the fast forward.)  -inf on some keys, on a whole query row, on every kept key; +inf and NaN (of either sign) at a kept
    and at a masked key; the lowest finite value on a whole row: zero rows, NaN rows and values are those
    of the generic kernels, forward and backward."""

    q, k, v, mask, bias, dout = make_case(dtype, prefix=(1,), rows=400, cols=133, head=32, masked=False, seed=9)
    inf, nan = float("inf"), float("nan")
    mask = torch.ones(1, 400, 133, dtype=torch.bool)
    mask[..., 100:] = False
    bias[0, 0, 0, 3, ::2] = -inf
    bias[0, 0, 0, 5] = -inf
    bias[0, 0, 0, 6, :100] = -inf
    bias[0, 0, 0, 7, 9] = inf
    bias[0, 0, 0, 8, 70] = nan
    bias[0, 0, 0, 9, 70] = -torch.tensor(nan)
    bias[0, 0, 0, 10, 120] = nan
    bias[0, 0, 0, 11] = torch.finfo(dtype).min
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v, bias)]
    m = mask.to(DEV) if masked else None

    def run():
        out = triangle_attention(leaves[0], leaves[1], leaves[2], m, leaves[3])
        return (out, *torch.autograd.grad(out, leaves, dout.to(DEV)))

    got = run()
    with _core.force_generic():
        want = run()
    rows = [i for i in range(133) if i not in (7, 8, 9, 10)]
    nan_rows = (7, 8, 9) if masked else (7, 8, 9, 10)
    for i in nan_rows:  # out is (1, rows, queries, heads, d)
        assert got[0][0, :, i, 0].isnan().all() and want[0][0, :, i, 0].isnan().all()
    assert (got[0][0, :, 5, 0] == 0).all()
    tol = dict(rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(got[0][:, :, rows], want[0][:, :, rows], **tol)
    torch.testing.assert_close(got[1][:, :, rows], want[1][:, :, rows], **tol)
    torch.testing.assert_close(got[4][..., rows, :], want[4][..., rows, :], rtol=2e-2, atol=0.1)  # (400 rows summed)
    for a, b in zip(got[2:4], want[2:4]):  # dK, dV of head 0 are NaN at every kept key, head 1 is finite
        torch.testing.assert_close(a[..., 1, :], b[..., 1, :], **tol)
        assert (a[..., 0, :].isnan() == b[..., 0, :].isnan()).all()
