"""16-bit pairs whose side is no multiple of 8, worked on a padded side: against the oracle at the criteria
of the other triangle multiplication tests, and against the unpadded kernels."""

import importlib

import pytest
import torch

from oops_amd import triangle_multiplication

from test_trimul_gpu import _check, _params

pytestmark = pytest.mark.gpu

DEV = "cuda"
mod = importlib.import_module("oops_amd.pair.triangle_multiplication")


@pytest.mark.parametrize(
    "dtype,c,h,n,direction,masked",
    [
        (torch.bfloat16, 128, 128, 99, "outgoing", True),
        (torch.float16, 64, 64, 97, "incoming", False),
        (torch.bfloat16, 128, 32, 105, "incoming", True),
        (torch.bfloat16, 32, 128, 100, "outgoing", False),
        (torch.float16, 120, 64, 98, "outgoing", True),
    ],
)
def test_against_oracle(dtype, c, h, n, direction, masked):
    g = torch.Generator().manual_seed(n)
    pair = torch.randn(1, n, n, c, generator=g).to(dtype).to(DEV).requires_grad_(True)
    mask = torch.rand(1, n, n, generator=g).to(DEV).requires_grad_(True) if masked else None
    weights, bs = _params(dtype, c, h, seed=n, biases=n % 2 == 1)
    assert mod._padded_side(n, pair.reshape(1, n * n, c), h) % 8 == 0
    _check(pair, mask, weights, bs, direction, dtype, mask_grad=masked)


@pytest.mark.parametrize("offset", [0, 3])
def test_against_unpadded(monkeypatch, offset):
    """Every output and gradient against the unpadded kernels (the same roundings), the pair on and off a
    16-byte boundary, the gradient too."""

    n, c, dtype = 109, 64, torch.bfloat16
    g = torch.Generator().manual_seed(1)
    flat = torch.randn(n * n * c + 8, generator=g).to(dtype).to(DEV)
    dflat = torch.randn(n * n * c + 8, generator=g).to(dtype).to(DEV)
    pair = flat[offset : offset + n * n * c].view(1, n, n, c).requires_grad_(True)
    dout = dflat[offset : offset + n * n * c].view(1, n, n, c)
    mask = torch.rand(1, n, n, generator=g).to(DEV).requires_grad_(True)
    weights, bs = _params(dtype, c, c, seed=2, biases=True)
    names = mod._WEIGHT_NAMES + mod._BIAS_NAMES
    kwargs = dict(zip(names, (*weights, *bs)))
    leaves = [pair, mask, *(t for t in kwargs.values() if t.requires_grad)]

    def run(d):
        out = triangle_multiplication(pair, mask, direction="outgoing", **kwargs)
        return (out, *torch.autograd.grad(out, leaves, d))

    got = run(dout)
    monkeypatch.setattr(mod, "_padded_side", lambda n, *a: n)
    want = run(dout.clone())
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype
        err = (a.float() - b.float()).norm() / b.float().norm()
        # one rounding of bfloat16 intermediates differs at most where a library GEMM sums in another order
        assert err <= 2.0**-8, float(err)


@pytest.mark.parametrize("eps", [0.0, 1e-50, 1e-12])
def test_small_output_eps(eps):
    """An output LayerNorm without (or with an all but vanishing) eps: no cell of the pair has equal channels, so
    every value is finite, as on the unpadded kernels."""

    n, c, dtype = 101, 64, torch.bfloat16
    g = torch.Generator().manual_seed(3)
    pair = torch.randn(1, n, n, c, generator=g).to(dtype).to(DEV).requires_grad_(True)
    dout = torch.randn(1, n, n, c, generator=g).to(dtype).to(DEV)
    weights, bs = _params(dtype, c, c, seed=4, biases=True)
    kwargs = dict(zip(mod._WEIGHT_NAMES + mod._BIAS_NAMES, (*weights, *bs)))
    leaves = [pair, *(t for t in kwargs.values() if t.requires_grad)]

    def run(e):
        out = triangle_multiplication(pair, None, direction="outgoing", output_norm_eps=e, **kwargs)
        return (out, *torch.autograd.grad(out, leaves, dout))

    for a, b in zip(run(eps), run(1e-10)):  # (1e-10 is nothing beside the variances here)
        assert bool(a.isfinite().all())
        assert (a.float() - b.float()).norm() <= 2.0**-8 * b.float().norm()
