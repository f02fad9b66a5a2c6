"""The float32 attention kernels at the edges of their 32-row tiles and 128-row blocks, for each head size
class, bias layout and mask, against the float64 oracle at the float32 criterion of accuracy.py."""

import pytest
import torch

from oops_amd import _lib, pair_bias_attention, triangle_attention
from oops_amd.attention import _core

from test_triangle_gpu import make_case, run_and_check

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("bias_kind", ["none", "shared", "full"])
@pytest.mark.parametrize("cols,head,layout", [(1, 32, "dense"), (31, 4, "dense"), (32, 32, "swapped"), (33, 24, "dense"),
                                              (65, 64, "swapped"), (127, 32, "dense"), (129, 36, "swapped"),
                                              (193, 32, "swapped")])  # fmt: skip
def test_tile_edges(cols, head, layout, bias_kind):
    case = make_case(torch.float32, prefix=(2,), rows=3, cols=cols, head=head, bias_kind=bias_kind, layout=layout,
                     masked=cols % 2 == 1, seed=cols)  # fmt: skip
    run_and_check(*case, torch.float32)


@pytest.mark.parametrize("cols,head", [(129, 32), (65, 24), (40, 64)])
def test_single_group(cols, head):
    """A shared bias of one row: its gradient is written by the dQ kernel."""

    case = make_case(torch.float32, prefix=(2,), rows=1, cols=cols, head=head, seed=cols)
    run_and_check(*case, torch.float32)


def test_masked_tiles():
    """Fully kept, fully masked and mixed 32-key tiles, a fully masked row, many rows per dBias part."""

    q, k, v, mask, bias, dout = make_case(torch.float32, prefix=(1,), rows=70, cols=150, head=32, seed=21)
    mask[:] = True
    mask[0, 0, 32:64] = False
    mask[0, 1, 5] = False
    mask[0, 2, :] = False
    mask[0, 3, 100:] = False
    run_and_check(q, k, v, mask, bias, dout, torch.float32)


@pytest.mark.parametrize("bias_kind", ["shared", "full"])
def test_nonfinite_as_generic(bias_kind):
    """inf and NaN in masked K and V rows, -inf, +inf and NaN biases: as the generic kernels, bit for bit where
    the result is finite up to the order of float32 sums."""

    q, k, v, mask, bias, dout = make_case(torch.float32, prefix=(1,), rows=3, cols=133, head=32, bias_kind=bias_kind,
                                          masked=False, seed=9)  # fmt: skip
    mask = torch.ones(1, 3, 133, dtype=torch.bool)
    mask[..., 100:] = False
    k[..., 101, :, :] = float("inf")
    v[..., 102, :, :] = float("nan")
    bias[..., 0, 3, ::2] = float("-inf")
    bias[..., 0, 5, :] = float("-inf")
    bias[..., 0, 6, 7] = float("inf")
    bias[..., 0, 7, 64] = float("nan")
    bias[..., 0, 8, 120] = float("nan")  # at a masked key
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v, bias)]

    def run():
        out = triangle_attention(leaves[0], leaves[1], leaves[2], mask.to(DEV), leaves[3])
        return (out, *torch.autograd.grad(out, leaves, dout.to(DEV)))

    got = run()
    with _core.force_generic():
        want = run()
    for g_, w in zip(got[:4], want[:4]):
        torch.testing.assert_close(g_, w, rtol=1e-5, atol=1e-5, equal_nan=True)
    # (dBias of the masked keys in a NaN row: not compared, tiles of masked keys only are skipped)
    torch.testing.assert_close(got[4][..., :100], want[4][..., :100], rtol=1e-5, atol=1e-5, equal_nan=True)


def test_rectangular_misaligned_bias_and_partial_gradients():
    """Fewer queries than keys, a bias view at an odd offset, gradients of k and the bias only."""

    g = torch.Generator().manual_seed(3)
    q = torch.randn(2, 3, 2, 45, 32, generator=g).to(DEV)
    k, v = (torch.randn(2, 3, 2, 171, 32, generator=g).to(DEV) for _ in range(2))
    bias = torch.randn(2, 1, 2, 45, 180, generator=g).to(DEV)[..., 3:174]
    dout = torch.randn(2, 3, 2, 45, 32, generator=g).to(DEV)
    k.requires_grad_(True)
    bias = bias.requires_grad_(True)

    def run():
        out = pair_bias_attention(q, k, v, None, bias)
        return (out, *torch.autograd.grad(out, (k, bias), dout))

    got = run()
    with _core.force_generic():
        want = run()
    for g_, w in zip(got, want):
        torch.testing.assert_close(g_, w, rtol=1e-5, atol=1e-5)


def test_single_group_phases():
    """A call for the shared dBias alone (no dQ) writes it, though the dQ kernel would when both are asked."""

    q, k, v, _, bias, dout = make_case(torch.float32, prefix=(1,), rows=1, cols=129, head=32, masked=False, seed=6)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v, bias)]
    out = triangle_attention(*leaves[:3], None, leaves[3])
    want = torch.autograd.grad(out, leaves[3], dout.to(DEV), retain_graph=True)[0]
    junk = torch.full((1 << 22,), 7.0, device=DEV)  # (what the allocator hands out next)
    del junk
    with _core.profile_phases(_lib.PHASE_DELTA | _lib.PHASE_DBIAS):
        got = torch.autograd.grad(out, leaves[3], dout.to(DEV))[0]
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_sample_without_bias(dtype):
    """A table whose first sample has no bias beside a biased one, forward and backward, against calls of its own."""

    s, n, h, d = 3, 72, 2, 32
    q, k, v, mask, bias, dout = make_case(dtype, prefix=(2,), rows=s, cols=n, heads=h, head=d, masked=False, seed=8)
    q, k, v, bias, dout = (t.to(DEV) for t in (q, k, v, bias, dout))
    per_b, st = s * n * h * d, (n * h * d, d, h * d)
    table, lse = [], s * h * n
    for b in range(2):
        qs = (b * per_b, *st)
        biased = dict(bias=(h * n * n, 0, n * n, n), dbias=(0, 0, n * n, n), bias_mode=_lib.BIAS_SHARED) if b else {}
        table += _core.table_row(groups=s, len_q=n, len_k=n, q=qs, k=qs, v=qs, lse_off=b * lse, **biased)
    scale = d**-0.5
    out, lo, l = _core._forward_impl(q, k, v, None, bias, table, h, scale, 2 * lse, True)
    dq, dk, dv, db = _core._backward_impl(dout, q, k, v, None, bias, out, lo, l, table, h, scale, h * n * n,
                                         [True] * 4)
    for b in range(2):
        leaves = [t[b : b + 1].clone().requires_grad_(True) for t in ((q, k, v, bias) if b else (q, k, v))]
        ref = triangle_attention(*leaves[:3], None, leaves[3] if b else None)
        grads = torch.autograd.grad(ref, leaves, dout[b : b + 1])
        tol = dict(rtol=1e-4, atol=1e-4) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-2)
        for x, y in zip((out, dq, dk, dv), (ref, *grads)):
            torch.testing.assert_close(x[b : b + 1], y, **tol)
        if b:
            torch.testing.assert_close(db.view(h, n, n), grads[3].view(h, n, n).float(), **tol)
