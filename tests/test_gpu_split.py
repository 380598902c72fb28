"""The split-operand GEMM kernel (bf16 parts of fp32 values) at the edges of its tiles, its
loaders and its reduction, against float64, and its infinities and NaN against fp32 arithmetic."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

EPS = 2.0**-24


def bound(K, absum, squares):
    """Error of a K-term sum from the kernel: one rounding per 32-wide k tile (plus four for the
    split-K partials and the epilogue) of sums no larger than the sum of magnitudes, one for the
    omitted parts of the products (below 2^-24 of each), one for the truncation of the k tiles'
    sums and one for each squared operand."""
    return (K / 32 + 6 + squares) * EPS * absum + 1e-37


def check(got, ref, absum, K, squares, what):
    err = (got.double() - ref).abs()
    over = (err / bound(K, absum, squares)).max().item()
    assert over <= 1.0, f"{what}: {over:.3g} of the bound"


def inputs(shape, gen, scale=1.0):
    return scale * torch.randn(*shape, generator=gen, device="cuda"), torch.rand(*shape, generator=gen, device="cuda") + 0.01


# widths 4 and up, one under and over the 16/32/64/128 tile sides and the 32-wide k tiles,
# rows of every alignment, reductions of one tile and of many
LINEAR = [(1, 5, 4), (64, 32, 64), (4095, 31, 1025), (8130, 33, 127), (2057, 100, 1029), (40001, 255, 61),
          (31, 4096, 1030), (515, 517, 1027), (2050, 64, 516), (96, 2052, 700), (99999, 39, 11), (16385, 7, 769),
          (769, 50001, 4), (5, 2048, 8193)]


@pytest.mark.parametrize("M,K,N", LINEAR)
def test_linear(M, K, N):
    from triton_tagi_amd.layers import Linear

    torch.manual_seed(M + K + N)
    gen = torch.Generator("cuda").manual_seed(7 * M + K + N)
    layer = Linear(K, N, device="cuda")
    ma, Sa = inputs((M, K), gen)
    dm, dS = inputs((M, N), gen)
    dS = -dS
    mz, Sz = layer.forward(ma, Sa)
    m0, S0 = layer.forward(ma, None)
    layer.forward(ma, Sa)
    d_ma, d_Sa = layer.backward(dm, dS)
    a, S, w, V, b, Vb, d, e = (t.double() for t in (ma, Sa, layer.mw, layer.Sw, layer.mb, layer.Sb, dm, dS))
    check(mz, a @ w + b, a.abs() @ w.abs() + b.abs(), K, 0, "mz")
    var = a**2 @ V + S @ (w**2 + V) + Vb
    check(Sz, var, var, 2 * K, 2, "Sz")
    check(m0, a @ w + b, a.abs() @ w.abs() + b.abs(), K, 0, "mz of a fixed input")
    check(S0, a**2 @ V + Vb, a**2 @ V + Vb, K, 1, "Sz of a fixed input")
    check(d_ma, d @ w.T, d.abs() @ w.abs().T, N, 0, "d_ma")
    check(d_Sa, e @ (w**2).T, e.abs() @ (w**2).T, N, 1, "d_Sa")
    check(layer.delta_mw, V * (a.T @ d), V * (a.abs().T @ d.abs()), M, 1, "delta_mw")
    check(layer.delta_Sw, V**2 * ((a**2).T @ e), V**2 * ((a**2).T @ e.abs()), M, 3, "delta_Sw")
    check(layer.delta_mb, Vb * d.sum(0, keepdim=True), Vb * d.abs().sum(0, keepdim=True), M, 1, "delta_mb")
    check(layer.delta_Sb, Vb**2 * e.sum(0, keepdim=True), Vb**2 * e.abs().sum(0, keepdim=True), M, 2, "delta_Sb")


# channels in and out of every alignment, taps that straddle k tiles, one-tap kernels, strides,
# images whose pixels do not fill a k tile
CONV = [(3, 32, 8, 64, 3, 1), (33, 64, 17, 80, 3, 1), (29, 13, 31, 138, 5, 1), (97, 37, 27, 65, 3, 2), (64, 64, 31, 17, 1, 1),
        (55, 5, 32, 66, 3, 1), (116, 30, 28, 70, 3, 2), (57, 96, 14, 133, 2, 2), (32, 32, 32, 48, 3, 1), (40, 48, 16, 96, 5, 2)]


@pytest.mark.parametrize("B,C,H,Cout,k,s", CONV)
def test_conv(B, C, H, Cout, k, s):
    from triton_tagi_amd.layers import Conv2D

    torch.manual_seed(B + C + H + Cout)
    gen = torch.Generator("cuda").manual_seed(B * C + H + Cout)
    layer = Conv2D(C, Cout, k, stride=s, padding=k // 2, device="cuda")
    ma, Sa = inputs((B, C, H, H), gen)
    mz, Sz = layer.forward(ma, Sa)
    dm, dS = inputs(tuple(mz.shape), gen)
    d_ma, d_Sa = layer.backward(dm, -dS)
    p = k // 2
    W, V = (t.double().T.reshape(Cout, C, k, k) for t in (layer.mw, layer.Sw))
    a, S, d, e = (t.double() for t in (ma, Sa, dm, -dS))
    b, Vb = layer.mb.double().view(1, -1, 1, 1), layer.Sb.double().view(1, -1, 1, 1)
    conv = lambda x, w: F.conv2d(x, w, stride=s, padding=p)  # noqa: E731
    back = lambda g, w: torch.nn.grad.conv2d_input(a.shape, w, g, stride=s, padding=p)  # noqa: E731
    wgr = lambda x, g: torch.nn.grad.conv2d_weight(x, W.shape, g, stride=s, padding=p).reshape(Cout, -1).T  # noqa: E731
    K = C * k * k
    check(mz, conv(a, W) + b, conv(a.abs(), W.abs()) + b.abs(), K, 0, "mz")
    var = conv(a**2, V) + conv(S, W**2 + V) + Vb
    check(Sz, var, var, 2 * K, 2, "Sz")
    check(d_ma, back(d, W), back(d.abs(), W.abs()), Cout * k * k, 0, "d_ma")
    check(d_Sa, back(e, W**2), back(e.abs(), W**2), Cout * k * k, 1, "d_Sa")
    Vw, M = layer.Sw.double(), d.numel() // Cout
    check(layer.delta_mw, Vw * wgr(a, d), Vw * wgr(a.abs(), d.abs()), M, 1, "delta_mw")
    check(layer.delta_Sw, Vw**2 * wgr(a**2, e), Vw**2 * wgr(a**2, e.abs()), M, 3, "delta_Sw")


@pytest.mark.parametrize("M,K,N", [(64, 64, 64), (3000, 100, 1130), (130, 700, 1001)])
def test_infinities_and_nan(M, K, N):
    """One infinite, one NaN and one huge operand: the outputs they reach are those of fp32
    arithmetic, the others are as without them."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(M + N)
    torch.manual_seed(M)
    layer = Linear(K, N, device="cuda")
    ma, Sa = inputs((M, K), gen)
    ma[1, 3], Sa[5, K - 1], ma[M - 1, 0], ma[7, 2] = float("inf"), float("nan"), 3e38, -3.4e38
    mz, Sz = layer.forward(ma, Sa)
    a, S, w, V = ma.cpu().float(), Sa.cpu().float(), layer.mw.cpu(), layer.Sw.cpu()
    rm = a @ w + layer.mb.cpu()
    rS = (a * a) @ V + S @ (w * w + V) + layer.Sb.cpu()
    for got, ref, what in ((mz.cpu(), rm, "mz"), (Sz.cpu(), rS, "Sz")):
        assert torch.equal(got.isnan(), ref.isnan()), what
        assert torch.equal(got.isinf(), ref.isinf()), what
        inf = ref.isinf()
        assert torch.equal(got[inf], ref[inf]), what
        fin = ref.isfinite()
        assert ((got[fin].double() - ref[fin].double()).norm() / ref[fin].double().norm()).item() < 1e-5, what


def test_sums_over_many_rows_are_unbiased():
    """Each output's error is below one rounding, but a shift common to all would add up where
    deltas are summed over the rows: it cancels between k tiles and between rows of tiles."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(3)
    torch.manual_seed(3)
    M, K, N = 32768, 512, 128
    layer = Linear(K, N, device="cuda")
    dm, dS = inputs((M, N), gen)
    layer.forward(*inputs((M, K), gen))
    d_ma, _ = layer.backward(dm, dS)
    err = d_ma.double() - dm.double() @ layer.mw.double().T
    # 2^24 outputs of independent roundings would leave 2^-12 of one rounding; the uncorrected
    # shift is 1e-8 of the outputs' size
    assert abs(err.mean().item()) < 1e-9 * d_ma.double().abs().mean().item()


@pytest.mark.parametrize("M", [1, 2, 4, 8, 15, 16])
def test_short_reductions(M):
    """Parameter deltas of few rows: an error within fp32 arithmetic's own bound, one rounding
    for each term and two for the variance's factor and its square."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(M)
    torch.manual_seed(M)
    K, N = 4096, 11008
    layer = Linear(K, N, device="cuda")
    for edge in (False, True):
        ma, Sa = inputs((M, K), gen)
        dm, dS = inputs((M, N), gen)
        if edge:  # values whose split parts are the largest: just below 1 + 2^-7
            ma, dm, dS = (1 + 2.0**-7 * (0.99 + 0.01 * torch.rand_like(t)) for t in (ma, dm, dS))
        layer.forward(ma, Sa)
        layer.backward(dm, dS)
        a, V, d, e = (t.double() for t in (ma, layer.Sw, dm, dS))
        for got, ref, mag, r in ((layer.delta_mw, V * (a.T @ d), V * (a.abs().T @ d.abs()), 1),
                                 (layer.delta_Sw, V**2 * ((a**2).T @ e), V**2 * ((a**2).T @ e.abs()), 3)):
            assert ((got.double() - ref).abs() / mag).max().item() < (M + r) * EPS


@pytest.mark.parametrize("K", [24, 500, 1003])
def test_constant_operands_leave_no_shift(K):
    """Weights that are all alike (an initial variance), at the value whose split leaves out
    the most: what is left out of the products averages out over the other operand."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(K)
    M, N = 8192, 256
    layer = Linear(K, N, bias=False, device="cuda")
    layer.mw.fill_(1.0077972)
    layer.Sw.fill_(1.0077972)
    ma, Sa = inputs((M, K), gen)
    for S in (Sa, None):
        mz, Sz = layer.forward(ma, S)
        w = layer.Sw.double()
        ref = ma.double() ** 2 @ w + (0 if S is None else S.double() @ (w * w + w))
        # columns alike: one number per row. A quarter of a rounding, three standard deviations
        # of the mean of M rows' own roundings (K / 32 of them, up to one each), and the half
        # that fp32 itself may round the constant mw^2 + Sw by
        shift = ((Sz.double() - ref) / ref).mean().item()
        own = 0.0 if S is None else 0.5
        assert abs(shift) < EPS * (0.25 + own + 3 * (K / 32 + 2) ** 0.5 / M**0.5)


@pytest.mark.parametrize("scale", [2.0**-90, 2.0**-105, 2.0**-112, 2.0**-120])
def test_small_values(scale):
    """Operands down to 2^-109 are split exactly; below, each is held to 2^-133."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(5)
    torch.manual_seed(5)
    M, K, N = 1000, 500, 516
    layer = Linear(K, N, bias=False, device="cuda")
    ma, Sa = inputs((M, K), gen, scale)
    Sa *= scale
    mz, Sz = layer.forward(ma, Sa)
    a, S, w, V = (t.double() for t in (ma, Sa, layer.mw, layer.Sw))
    fine = 2.0**-133  # per operand value, times the other operand
    err = (mz.double() - a @ w).abs()
    assert (err <= bound(K, a.abs() @ w.abs(), 0) + fine * w.abs().sum(0)).all()
    err = (Sz.double() - (a**2 @ V + S @ (w**2 + V))).abs()
    assert (err <= bound(2 * K, a**2 @ V + S @ (w**2 + V), 2) + fine * (2 * V + w**2).sum(0) + 2.0**-126).all()
