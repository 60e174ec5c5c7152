"""GPU tests of the kernels whose FP32 products run as split bf16 MFMAs
(three bf16 pieces a value, six products): sizes at the edges of their tiles
and of their cuts of the work, against float64, with the bound that the
splitting and the FP32 accumulators give, and infinities and NaN."""
import numpy as np
import pytest
import torch

import cxxgpt_attn as cx

pytestmark = pytest.mark.gpu


def gemm_bound(a, b):
    """|C - C64| for C = a b: sums of K products through FP32 accumulators, at
    most two roundings for each 16-wide step (one product's pieces and
    alignment in the matrix unit, one into the accumulator), plus the dropped
    terms and the joining of pieces: (K / 8 + 16) 2^-24 of sum |a||b|."""
    return (a.shape[1] / 8 + 16) * 2.0 ** -24 * (a.abs() @ b.abs())


def check(got, a, b, name, ref=None):
    want = a @ b if ref is None else ref
    err = (got.double() - want).abs()
    lim = gemm_bound(a, b) + 1e-30
    assert bool((err <= lim).all()), f"{name}: {(err / lim).max().item():.2f} of the bound"


# rows: below, at and past the 128- and 256-row tiles; widths: k-tails of 4 and
# 28 floats, column remainders; products of one run a tile, of several runs a
# tile, and (the last two) of equal runs that cut tiles unevenly
@pytest.mark.parametrize("M,E,F", [(1, 4, 8), (53, 36, 132), (127, 64, 60), (129, 260, 1028),
                                   (257, 132, 388), (300, 768, 2052), (1160, 572, 2288)])
def test_ffn_products(dev, M, E, F):
    g = torch.Generator(device=dev).manual_seed(M + E)
    X, dY = (torch.randn(M, E, device=dev, generator=g) for _ in range(2))
    W1, W2 = (torch.randn(*s, device=dev, generator=g) for s in ((F, E), (E, F)))
    pre, act = torch.empty(M, F, device=dev), torch.empty(M, F, device=dev)
    Y, dX = torch.empty(M, E, device=dev), torch.empty(M, E, device=dev)
    dW1, dW2 = torch.zeros(F, E, device=dev), torch.zeros(E, F, device=dev)
    cx.ffn_fwd(X, W1, W2, pre, act, Y, M, E, F)
    # gelu'(0) = 1/2 exactly: dact = (dY W2) / 2
    cx.ffn_bwd(X, W1, W2, act, torch.zeros_like(act), dY, dX, dW1, dW2, M, E, F)
    x, w1, w2, dy, a = (t.double() for t in (X, W1, W2, dY, act))
    check(pre, x, w1.t(), "pre")
    check(Y, a, w2.t(), "Y")
    check(dW2, dy.t(), a, "dW2")
    da = dy @ w2 / 2
    # dact itself carries its product's error, which the next products scale
    e = gemm_bound(dy, w2) / 2
    for got, want, lim, n in ((dX, da @ w1, gemm_bound(da, w1) + e @ w1.abs(), "dX"),
                              (dW1, da.t() @ x, gemm_bound(da.t(), x) + e.t() @ x.abs(), "dW1")):
        assert bool(((got.double() - want).abs() <= lim).all()), n


@pytest.mark.parametrize("M,E,F", [(40, 128, 64), (300, 96, 520)])
def test_ffn_non_finite(dev, M, E, F):
    """An infinity or NaN in an operand gives the FP32 product's own pattern."""
    g = torch.Generator(device=dev).manual_seed(3)
    X, W1 = torch.randn(M, E, device=dev, generator=g), torch.randn(F, E, device=dev, generator=g)
    W2 = torch.zeros(E, F, device=dev)
    X[1, 5], X[7, 0], X[M - 1, E - 1], W1[3, 2], X[9, 9] = np.inf, -np.inf, np.nan, np.inf, 3.4e38
    # 3.4e38 / 2 is finite; beside W1's infinity the product must not overflow to
    # the other one, which float64 would not show
    W1[0, 9] = W1[3, 9] = 0.5
    pre, act, Y = (torch.empty(M, n, device=dev) for n in (F, F, E))
    cx.ffn_fwd(X, W1, W2, pre, act, Y, M, E, F)
    want = (X.double() @ W1.double().t()).float()   # overflow to inf as in FP32
    big = want.abs() > 3.3e38   # sums within rounding of the overflow threshold
    assert torch.equal(torch.isnan(pre), torch.isnan(want))
    inf = torch.isinf(want) & ~big | torch.isinf(X.double() @ W1.double().t())
    assert torch.equal(pre[inf], want[inf])
    assert bool(torch.isfinite(pre[torch.isfinite(want) & ~big]).all())
