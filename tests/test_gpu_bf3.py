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


def heads(t, B, S, H, Dh):
    return t.double().view(B, S, H, Dh).permute(0, 2, 1, 3).reshape(B * H, S, Dh)


def flat(t, B, S, H, Dh):
    return t.view(B, H, S, Dh).permute(0, 2, 1, 3).reshape(B * S, H * Dh)


def mha64(Q, K, V, dO, B, S, H, Dh):
    """float64 causal attention, its row statistics and gradients, and a bound
    on each one's FP32 error: a score q.k is off by at most (Dh / 8 + 16) 2^-24
    of sum |q||k| (gemm_bound), lse by as much, so P by twice that relatively
    (plus the exponential's 2^-22), and the sums over rows by (S / 8 + 16) 2^-24
    of their terms' magnitudes."""
    q, k, v, do = (heads(t, B, S, H, Dh) for t in (Q, K, V, dO))
    T = lambda t: t.transpose(1, 2).contiguous()   # noqa: E731
    scale = Dh ** -0.5
    future = torch.ones(S, S, device=q.device, dtype=torch.bool).triu_(1)
    s = (torch.bmm(q, T(k)) * scale).masked_fill_(future, -np.inf)
    lse = torch.logsumexp(s, 2)
    p = torch.exp(s - lse.unsqueeze(2))
    o = torch.bmm(p, v)
    di = (do * o).sum(2, keepdim=True)
    ds = (torch.bmm(do, T(v)) - di) * p * scale
    out = [o, torch.bmm(ds, k), torch.bmm(T(ds), q), torch.bmm(T(p), do)]
    es = (Dh / 8 + 16) * 2.0 ** -24 * (torch.bmm(q.abs(), T(k.abs())) * scale).masked_fill_(future, 0)
    e = 2 * es.amax(2, keepdim=True) + 2.0 ** -22 + (S / 8 + 16) * 2.0 ** -24
    pe = p * e
    we = p * (torch.bmm(do.abs(), T(v.abs())) + (do * o).abs().sum(2, keepdim=True)) * scale * e * 2
    lim = [torch.bmm(pe, v.abs()), torch.bmm(we, k.abs()), torch.bmm(T(we), q.abs()),
           torch.bmm(T(pe), do.abs())]
    return ([flat(t, B, S, H, Dh) for t in out] + [lse],
            [flat(t, B, S, H, Dh) for t in lim] + [e.squeeze(2)])


def within(got, want, lim, name):
    err = (got.double() - want).abs() / (lim + 1e-12)
    assert bool(torch.isfinite(got).all()) and err.max().item() <= 1.0, f"{name}: {err.max().item()}"


# (B, S, H, Dh): each kernel at the edges of its 32- and 64-row tiles, of its
# column steps (Dh 20 .. 96) and of its rule (64-row tiles against 256 units):
# one round, one to two, many; rows past S in the last tile
@pytest.mark.parametrize("B,S,H,Dh", [
    (2, 96, 3, 20), (1, 127, 4, 32), (3, 161, 2, 36), (1, 128, 5, 64), (2, 321, 3, 64),
    (2, 65, 2, 68), (1, 333, 3, 80), (2, 31, 2, 96), (1, 193, 4, 92),
    (8, 300, 8, 64), (8, 257, 15, 36), (16, 257, 9, 64), (16, 290, 8, 24)])
@pytest.mark.parametrize("use_lse", [True, False])
def test_mha_split(dev, B, S, H, Dh, use_lse):
    g = torch.Generator(device=dev).manual_seed(S * Dh)
    Q, K, V, dO = (torch.randn(B * S, H * Dh, device=dev, generator=g) for _ in range(4))
    Q[: S // 2] *= 6.0   # scores that move the softmax reference between tiles
    O, dQ, dK, dV = (torch.full_like(Q, np.nan) for _ in range(4))
    lse = torch.empty(B * H, S, device=dev) if use_lse else None
    cx.mha_fwd(Q, K, V, O, B, S, H, Dh, lse=lse)
    cx.mha_bwd(Q, K, V, O, dO, dQ, dK, dV, B, S, H, Dh, lse=lse)
    want, lim = mha64(Q, K, V, dO, B, S, H, Dh)
    for got, w, e, n in zip((O, dQ, dK, dV, lse), want, lim, ("O", "dQ", "dK", "dV", "lse")):
        if got is not None:
            within(got, w, e, n)


@pytest.mark.parametrize("B,S,H,Dh", [(1, 160, 2, 64), (1, 100, 2, 96), (16, 257, 9, 64)])
def test_mha_minus_infinite_scores(dev, B, S, H, Dh):
    """A key whose scores are all -inf has probability 0, as in FP32."""
    g = torch.Generator(device=dev).manual_seed(9)
    Q, K, V = (torch.randn(B * S, H * Dh, device=dev, generator=g) for _ in range(3))
    Q[:, 0] = Q[:, 0].abs() + 0.5
    K.view(B, S, -1)[:, 3::7, 0] = -np.inf   # head 0; never a sequence's first key
    O = torch.empty_like(Q)
    cx.mha_fwd(Q, K, V, O, B, S, H, Dh)
    fin = K.clamp(min=-1e3)   # scores below -60 of the others': probability 0 to FP32 as well
    want, lim = mha64(Q, fin, V, V, B, S, H, Dh)
    rows = heads(K, B, S, H, Dh).isfinite().all(2, keepdim=True)
    assert bool(torch.isfinite(O).all())
    # the bound of the same products without the infinite keys
    lim = mha64(Q, torch.where(flat(rows.expand(-1, -1, Dh), B, S, H, Dh), K, torch.zeros_like(K)), V, V,
                B, S, H, Dh)[1]
    within(O, want[0], lim[0] * 4, "O")


# enough 64 x 64 tiles for the split products (more than 512 forward, 384
# backward), at row, key-step and column remainders; with and without the
# context, and the rotation
@pytest.mark.parametrize("api,B,S,D,E", [
    ("kattn", 65, 65, 80, 112), ("rope", 65, 65, 80, 112), ("kattn", 24, 190, 208, 208),
    ("rope", 24, 190, 208, 208), ("lin_elu", 24, 190, 208, 208), ("kattn", 90, 33, 352, 144),
    ("rope", 90, 33, 352, 144)])
def test_linear_tiles(dev, api, B, S, D, E):
    g = torch.Generator(device=dev).manual_seed(B + S)
    Q, K = (torch.randn(B * S, D, device=dev, generator=g) for _ in range(2))
    V, dO = (torch.randn(B * S, E, device=dev, generator=g) for _ in range(2))
    O, dV = torch.full_like(V, np.nan), torch.full_like(V, np.nan)
    dQ, dK = torch.full_like(Q, np.nan), torch.full_like(Q, np.nan)
    den = torch.empty(B * S, device=dev)
    n = cx.lin_ctx_size(B, S, D, E)
    ctx = torch.empty(n // 4, device=dev) if n else None
    q, k = (t.double().view(B, S, D) for t in (Q, K))
    if api == "rope":
        w = torch.tensor([10000.0 ** (-2 * i / D) for i in range(D // 2)], device=dev)
        a = (torch.arange(S, device=dev).float()[:, None] * w).double()

        def rot(x, s):
            y = torch.empty_like(x)
            c, t = torch.cos(a), s * torch.sin(a)
            y[..., 0::2] = x[..., 0::2] * c - x[..., 1::2] * t
            y[..., 1::2] = x[..., 0::2] * t + x[..., 1::2] * c
            return y
        q, k = rot(q, 1), rot(k, 1)
        cx.kattn_rope_fwd(Q, K, V, O, den, B, S, D, E, ctx=ctx)
        cx.kattn_rope_bwd(Q, K, V, O, dO, den, dQ, dK, dV, B, S, D, E, ctx=ctx)
    elif api == "kattn":
        cx.kattn_fwd(Q, K, V, O, den, None, None, None, B, S, D, E)
        cx.kattn_bwd(Q, K, V, O, dO, den, dQ, dK, dV, B, S, D, E)
    else:
        cx.lin_elu_fwd(Q, K, V, O, den, ctx, B, S, E)
        cx.lin_elu_bwd(Q, K, V, O, dO, den, dQ, dK, dV, B, S, E, ctx=ctx)
    T = lambda t: t.transpose(1, 2).contiguous()   # noqa: E731
    fq, fk = (torch.where(x > 0, x + 1, torch.exp(x)) for x in (q, k))
    v, do = V.double().view(B, S, E), dO.double().view(B, S, E)
    A = torch.bmm(fq, T(fk)).tril_()
    d = A.sum(2, keepdim=True) + 1e-8
    o = torch.bmm(A, v) / d
    dn, dd = do / d, -(do * o).sum(2, keepdim=True) / d
    G = (torch.bmm(dn, T(v)) + dd).tril_()
    gq, gk = torch.bmm(G, fk) * fq.clamp(max=1), torch.bmm(T(G), fq) * fk.clamp(max=1)
    # a score's error is (D / 8 + 16) 2^-24 of it (all terms positive), G's that
    # of its terms' magnitudes; the sums over rows add (S / 8 + 16) 2^-24; the
    # float angles of the rotation, up to S, 2^-24 S
    e = (max(D, E) / 8 + S / 8 + 40 + (4 * S if api == "rope" else 0)) * 2.0 ** -24
    H = (torch.bmm(dn.abs(), T(v.abs())) + (do * o).abs().sum(2, keepdim=True) / d).tril_() * e
    lq, lk = torch.bmm(H, fk) * fq.clamp(max=1), torch.bmm(T(H), fq) * fk.clamp(max=1)
    if api == "rope":
        gq, gk = rot(gq, -1), rot(gk, -1)
        lq, lk = (x.view(B, S, D // 2, 2).sum(3, keepdim=True).expand(-1, -1, -1, 2).reshape(B, S, D)
                  for x in (lq, lk))
    within(O, o.view(-1, E), (torch.bmm(A, v.abs()) / d).view(-1, E) * e * 2, "O")
    within(den, d.view(-1), d.view(-1) * e, "den")
    within(dV, torch.bmm(T(A), dn).view(-1, E), torch.bmm(T(A), dn.abs()).view(-1, E) * e * 2, "dV")
    within(dQ, gq.reshape(-1, D), lq.view(-1, D) * 2, "dQ")
    within(dK, gk.reshape(-1, D), lk.view(-1, D) * 2, "dK")
