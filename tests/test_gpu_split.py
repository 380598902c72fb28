"""The split-operand GEMM kernel (bf16 parts of fp32 values) at the edges of its tiles, its
loaders and its reduction, against float64, and its infinities and NaN against fp32 arithmetic.

The tables name the product and the tile that the planner gives a shape; each test checks that
it does, so that a change of the planner shows here as a tile no longer reached."""

import ctypes

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

EPS = 2.0**-24


def bound(K, absum, squares, split=True):
    """Error of a K-term sum from the split kernel: one rounding per 32-wide k tile (plus four for
    the split-K partials and the epilogue) of sums no larger than the sum of magnitudes, one for
    the omitted parts of the products (below 2^-24 of each), one for the truncation of the k
    tiles' sums and one for each squared operand. From the fp32 kernel, which a few of a layer's
    products run: one rounding for every term."""
    return ((K / 32 if split else K) + 6 + squares) * EPS * absum + 1e-37


def check(got, ref, absum, K, squares, what, plan=None):
    err = (got.double() - ref).abs()
    over = (err / bound(K, absum, squares, plan is None or plan.split_kernel)).max().item()
    assert over <= 1.0, f"{what}: {over:.3g} of the bound"


def inputs(shape, gen, scale=1.0):
    return scale * torch.randn(*shape, generator=gen, device="cuda"), torch.rand(*shape, generator=gen, device="cuda") + 0.01


OPS = ("fwd", "fwd0", "bwd", "wg")  # forward, of an input without variance, input deltas, parameter deltas


def linear_plan(op, M, K, N):
    from triton_tagi_amd import _lib

    p = _lib.Plan()
    _lib.call("tagi_linear_plan", OPS.index(op), M, K, N, -1, ctypes.byref(p))
    return p


def conv_plan(op, layer, B, H):
    from triton_tagi_amd import _lib

    p = _lib.Plan()
    geo = layer._geom(B, layer.C_in, H, H)
    _lib.call("tagi_conv2d_plan", OPS.index(op), geo, -1, ctypes.byref(p))
    return p


def runs_split(p, tile):
    assert p.split_kernel and (p.tile_rows, p.tile_cols) == tile, (p.split_kernel, p.tile_rows, p.tile_cols)


# every tile of every product, with rows that float4 loads divide and with others, remainders in
# rows, columns and the last k tile (found by asking the planner; the 128 x 64 and 128 x 128
# tiles of some products are only reached with the reduction cut up)
LINEAR_TILES = [
    ('bwd', (128, 128), 335, 8464, 12), ('bwd', (128, 32), 4912, 399, 18), ('bwd', (128, 32), 9090, 196, 20),
    ('bwd', (128, 64), 13923, 101, 25), ('bwd', (128, 64), 1282, 1364, 20), ('bwd', (256, 128), 26724, 213, 131),
    ('bwd', (256, 128), 58219, 84, 136), ('bwd', (256, 64), 49211, 33, 169), ('bwd', (256, 64), 51056, 40, 136),
    ('bwd', (32, 32), 508, 275, 242), ('bwd', (32, 32), 844, 184, 220), ('bwd', (64, 32), 10508, 73, 45),
    ('bwd', (64, 32), 10809, 88, 36), ('bwd', (64, 64), 2334, 329, 45), ('bwd', (64, 64), 1246, 620, 44),
    ('fwd', (128, 128), 68, 373, 8458), ('fwd', (128, 128), 69, 468, 5884), ('fwd', (128, 32), 26014, 17, 81),
    ('fwd', (128, 32), 24633, 20, 72), ('fwd', (128, 64), 1839, 2803, 143), ('fwd', (128, 64), 625, 1748, 444),
    ('fwd', (256, 128), 8926, 132, 708), ('fwd', (256, 64), 18997, 257, 37), ('fwd', (256, 64), 8471, 648, 36),
    ('fwd', (32, 32), 665, 177, 286), ('fwd', (32, 32), 657, 188, 272), ('fwd', (64, 32), 2174, 237, 73),
    ('fwd', (64, 32), 8511, 56, 72), ('fwd', (64, 64), 194, 193, 914), ('fwd', (64, 64), 3752, 44, 204),
    ('fwd0', (128, 128), 50170, 72, 100), ('fwd0', (128, 32), 52300, 25, 27), ('fwd0', (128, 32), 8423, 24, 200),
    ('fwd0', (128, 64), 50794, 73, 35), ('fwd0', (128, 64), 49600, 88, 36), ('fwd0', (256, 128), 54577, 140, 68),
    ('fwd0', (256, 64), 17914, 349, 33), ('fwd0', (256, 64), 8372, 808, 40), ('fwd0', (32, 32), 665, 177, 286),
    ('fwd0', (32, 32), 657, 188, 272), ('fwd0', (64, 32), 2174, 237, 73), ('fwd0', (64, 32), 8511, 56, 72),
    ('fwd0', (64, 64), 194, 193, 914), ('fwd0', (64, 64), 3752, 44, 204), ('wg', (128, 128), 8851, 1692, 68),
    ('wg', (128, 256), 1316, 65, 9177), ('wg', (128, 256), 2419, 72, 5460), ('wg', (32, 128), 21, 653, 2974),
    ('wg', (32, 128), 18, 532, 3808), ('wg', (32, 32), 175, 545, 354), ('wg', (32, 32), 143, 204, 1160),
    ('wg', (32, 64), 198, 65, 2678), ('wg', (32, 64), 201, 136, 1388), ('wg', (64, 128), 616, 6433, 71),
    ('wg', (64, 128), 11407, 392, 80), ('wg', (64, 256), 885, 35, 9201), ('wg', (64, 256), 1229, 32, 6684),
    ('wg', (64, 64), 194, 193, 914), ('wg', (64, 64), 199, 1332, 136),
]


@pytest.mark.parametrize("op,tile,M,K,N", LINEAR_TILES)
def test_linear_tiles(op, tile, M, K, N):
    runs_split(linear_plan(op, M, K, N), tile)
    test_linear(M, K, N)


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
    fwd, fwd0, bwd, wg = (linear_plan(op, M, K, N) for op in OPS)
    check(mz, a @ w + b, a.abs() @ w.abs() + b.abs(), K, 0, "mz", fwd)
    var = a**2 @ V + S @ (w**2 + V) + Vb
    check(Sz, var, var, 2 * K, 2, "Sz", fwd)
    check(m0, a @ w + b, a.abs() @ w.abs() + b.abs(), K, 0, "mz of a fixed input", fwd0)
    check(S0, a**2 @ V + Vb, a**2 @ V + Vb, K, 1, "Sz of a fixed input", fwd0)
    check(d_ma, d @ w.T, d.abs() @ w.abs().T, N, 0, "d_ma", bwd)
    check(d_Sa, e @ (w**2).T, e.abs() @ (w**2).T, N, 1, "d_Sa", bwd)
    check(layer.delta_mw, V * (a.T @ d), V * (a.abs().T @ d.abs()), M, 1, "delta_mw", wg)
    check(layer.delta_Sw, V**2 * ((a**2).T @ e), V**2 * ((a**2).T @ e.abs()), M, 3, "delta_Sw", wg)
    check(layer.delta_mb, Vb * d.sum(0, keepdim=True), Vb * d.abs().sum(0, keepdim=True), M, 1, "delta_mb", wg)
    check(layer.delta_Sb, Vb**2 * e.sum(0, keepdim=True), Vb**2 * e.abs().sum(0, keepdim=True), M, 2, "delta_Sb", wg)


CONV_TILES = [
    ('bwd', (128, 128), 127, 240, 14, 16, 1, 1), ('bwd', (128, 128), 132, 254, 20, 144, 1, 2),
    ('bwd', (128, 128), 61, 352, 11, 32, 2, 2), ('bwd', (128, 128), 76, 323, 11, 32, 2, 1),
    ('bwd', (128, 32), 46, 4, 36, 16, 3, 1), ('bwd', (128, 32), 34, 73, 27, 48, 1, 1),
    ('bwd', (128, 32), 85, 4, 14, 288, 3, 2), ('bwd', (128, 32), 75, 6, 17, 64, 3, 1),
    ('bwd', (128, 64), 78, 48, 28, 6, 3, 2), ('bwd', (128, 64), 182, 35, 11, 6, 3, 1),
    ('bwd', (128, 64), 55, 40, 31, 16, 1, 1), ('bwd', (128, 64), 10, 567, 37, 16, 1, 1),
    ('bwd', (128, 64), 177, 48, 11, 32, 2, 2), ('bwd', (128, 64), 23, 182, 29, 32, 1, 1),
    ('bwd', (256, 128), 142, 68, 9, 48, 5, 1), ('bwd', (256, 128), 59, 87, 34, 16, 3, 1),
    ('bwd', (256, 128), 80, 80, 35, 32, 3, 2), ('bwd', (256, 128), 30, 337, 24, 32, 2, 1),
    ('bwd', (256, 64), 190, 40, 17, 16, 3, 1), ('bwd', (256, 64), 32, 38, 22, 112, 3, 1),
    ('bwd', (256, 64), 149, 48, 25, 32, 3, 2), ('bwd', (32, 32), 13, 20, 23, 10, 5, 1),
    ('bwd', (32, 32), 13, 62, 17, 17, 3, 1), ('bwd', (32, 32), 15, 156, 10, 16, 3, 1),
    ('bwd', (32, 32), 12, 421, 4, 208, 3, 2), ('bwd', (32, 32), 11, 176, 11, 128, 2, 2),
    ('bwd', (32, 32), 4, 285, 9, 160, 3, 2), ('bwd', (64, 32), 47, 60, 10, 5, 5, 1),
    ('bwd', (64, 32), 24, 35, 18, 14, 3, 1), ('bwd', (64, 32), 63, 8, 22, 16, 3, 1),
    ('bwd', (64, 32), 166, 6, 18, 48, 3, 2), ('bwd', (64, 32), 26, 16, 18, 128, 3, 2),
    ('bwd', (64, 32), 2, 86, 29, 128, 2, 1), ('bwd', (64, 64), 13, 56, 34, 43, 2, 2),
    ('bwd', (64, 64), 20, 39, 9, 222, 3, 2), ('bwd', (64, 64), 45, 48, 22, 16, 3, 2),
    ('bwd', (64, 64), 3, 413, 30, 48, 1, 1), ('bwd', (64, 64), 90, 240, 6, 64, 1, 1),
    ('bwd', (64, 64), 134, 101, 9, 96, 2, 2), ('fwd', (128, 128), 88, 6, 17, 72, 3, 1),
    ('fwd', (128, 128), 172, 5, 12, 89, 3, 1), ('fwd', (128, 128), 123, 16, 11, 208, 1, 1),
    ('fwd', (128, 128), 50, 32, 23, 112, 1, 1), ('fwd', (128, 32), 165, 16, 19, 8, 2, 1),
    ('fwd', (128, 32), 125, 32, 23, 16, 1, 1), ('fwd', (128, 64), 113, 16, 10, 308, 1, 1),
    ('fwd', (128, 64), 152, 32, 9, 112, 1, 1), ('fwd', (256, 128), 76, 16, 12, 560, 3, 1),
    ('fwd', (256, 128), 67, 160, 15, 480, 1, 1), ('fwd', (256, 64), 58, 31, 19, 40, 3, 1),
    ('fwd', (256, 64), 19, 165, 20, 35, 2, 1), ('fwd', (256, 64), 109, 272, 13, 36, 1, 1),
    ('fwd', (256, 64), 26, 96, 18, 48, 3, 1), ('fwd', (32, 32), 1, 17, 30, 252, 3, 1),
    ('fwd', (32, 32), 6, 26, 38, 18, 3, 1), ('fwd', (32, 32), 3, 16, 18, 240, 3, 1),
    ('fwd', (32, 32), 7, 128, 9, 472, 1, 1), ('fwd', (64, 32), 12, 5, 7, 472, 5, 1),
    ('fwd', (64, 32), 4, 13, 18, 225, 3, 1), ('fwd', (64, 32), 21, 16, 38, 8, 3, 1),
    ('fwd', (64, 32), 154, 32, 12, 48, 1, 1), ('fwd', (64, 64), 18, 59, 4, 316, 2, 1),
    ('fwd', (64, 64), 4, 7, 13, 285, 5, 1), ('fwd', (64, 64), 19, 48, 14, 48, 2, 1),
    ('fwd', (64, 64), 27, 160, 13, 48, 1, 1), ('fwd0', (128, 128), 123, 16, 11, 208, 1, 1),
    ('fwd0', (128, 128), 50, 32, 23, 112, 1, 1), ('fwd0', (128, 32), 27, 6, 34, 20, 3, 1),
    ('fwd0', (128, 32), 6, 26, 38, 18, 3, 1), ('fwd0', (128, 32), 165, 16, 19, 8, 2, 1),
    ('fwd0', (128, 32), 71, 32, 27, 24, 1, 1), ('fwd0', (128, 64), 17, 35, 26, 92, 1, 1),
    ('fwd0', (128, 64), 14, 5, 37, 42, 3, 1), ('fwd0', (128, 64), 113, 16, 10, 308, 1, 1),
    ('fwd0', (128, 64), 152, 32, 9, 112, 1, 1), ('fwd0', (256, 128), 5, 135, 30, 72, 3, 1),
    ('fwd0', (256, 128), 73, 281, 7, 66, 2, 1), ('fwd0', (256, 128), 49, 16, 34, 80, 3, 1),
    ('fwd0', (256, 128), 92, 128, 25, 80, 1, 1), ('fwd0', (256, 64), 58, 31, 19, 40, 3, 1),
    ('fwd0', (256, 64), 50, 117, 14, 35, 2, 1), ('fwd0', (256, 64), 46, 16, 19, 48, 5, 1),
    ('fwd0', (256, 64), 26, 96, 18, 48, 3, 1), ('fwd0', (32, 32), 1, 17, 30, 252, 3, 1),
    ('fwd0', (32, 32), 4, 7, 13, 285, 5, 1), ('fwd0', (32, 32), 3, 16, 18, 240, 3, 1),
    ('fwd0', (32, 32), 7, 128, 9, 472, 1, 1), ('fwd0', (64, 32), 26, 3, 6, 500, 5, 1),
    ('fwd0', (64, 32), 11, 91, 10, 342, 1, 1), ('fwd0', (64, 32), 21, 16, 38, 8, 3, 1),
    ('fwd0', (64, 32), 154, 32, 12, 48, 1, 1), ('fwd0', (64, 64), 18, 59, 4, 316, 2, 1),
    ('fwd0', (64, 64), 55, 26, 4, 166, 3, 1), ('fwd0', (64, 64), 19, 48, 14, 48, 2, 1),
    ('fwd0', (64, 64), 5, 224, 12, 288, 1, 1), ('wg', (128, 128), 1, 577, 8, 221, 5, 2),
    ('wg', (128, 128), 195, 280, 7, 76, 2, 1), ('wg', (128, 128), 2, 520, 6, 244, 5, 2),
    ('wg', (128, 256), 31, 123, 10, 496, 5, 2), ('wg', (128, 256), 156, 64, 16, 416, 1, 1),
    ('wg', (128, 256), 11, 168, 11, 208, 5, 1), ('wg', (32, 128), 20, 12, 21, 591, 1, 1),
    ('wg', (32, 128), 175, 320, 7, 224, 1, 2), ('wg', (32, 128), 47, 16, 32, 560, 1, 2),
    ('wg', (32, 32), 8, 199, 5, 34, 5, 1), ('wg', (32, 32), 6, 100, 8, 140, 5, 2),
    ('wg', (32, 32), 2, 96, 15, 304, 3, 2), ('wg', (32, 64), 3, 490, 5, 289, 3, 2),
    ('wg', (32, 64), 3, 440, 8, 108, 5, 2), ('wg', (32, 64), 13, 12, 8, 268, 5, 1),
    ('wg', (64, 128), 6, 577, 4, 354, 3, 2), ('wg', (64, 128), 2, 504, 7, 368, 3, 2),
    ('wg', (64, 128), 2, 512, 8, 208, 5, 1), ('wg', (64, 256), 82, 37, 8, 197, 3, 1),
    ('wg', (64, 256), 168, 16, 8, 480, 5, 2), ('wg', (64, 256), 150, 96, 15, 416, 1, 2),
    ('wg', (64, 64), 4, 126, 7, 55, 5, 1), ('wg', (64, 64), 3, 392, 7, 212, 3, 2),
    ('wg', (64, 64), 3, 512, 15, 48, 3, 2),
]


@pytest.mark.parametrize("op,tile,B,C,H,Cout,k,s", CONV_TILES)
def test_conv_tiles(op, tile, B, C, H, Cout, k, s):
    """Every tile beside the loaders of whole k tiles per tap, of float4 and of element-wise
    patches, with remainders in rows and columns."""
    from triton_tagi_amd.layers import Conv2D

    layer = Conv2D(C, Cout, k, stride=s, padding=k // 2, device="cuda")
    runs_split(conv_plan(op, layer, B, H), tile)
    test_conv(B, C, H, Cout, k, s)


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
    m0, S0 = layer.forward(ma, None)
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
    fwd, fwd0, bwd, wg = (conv_plan(op, layer, B, H) for op in OPS)
    check(mz, conv(a, W) + b, conv(a.abs(), W.abs()) + b.abs(), K, 0, "mz", fwd)
    var = conv(a**2, V) + conv(S, W**2 + V) + Vb
    check(Sz, var, var, 2 * K, 2, "Sz", fwd)
    check(m0, conv(a, W) + b, conv(a.abs(), W.abs()) + b.abs(), K, 0, "mz of a fixed input", fwd0)
    check(S0, conv(a**2, V) + Vb, conv(a**2, V) + Vb, K, 1, "Sz of a fixed input", fwd0)
    check(d_ma, back(d, W), back(d.abs(), W.abs()), Cout * k * k, 0, "d_ma", bwd)
    check(d_Sa, back(e, W**2), back(e.abs(), W**2), Cout * k * k, 1, "d_Sa", bwd)
    Vw, M = layer.Sw.double(), d.numel() // Cout
    check(layer.delta_mw, Vw * wgr(a, d), Vw * wgr(a.abs(), d.abs()), M, 1, "delta_mw", wg)
    check(layer.delta_Sw, Vw**2 * wgr(a**2, e), Vw**2 * wgr(a**2, e.abs()), M, 3, "delta_Sw", wg)


def same_specials(got, ref, what):
    """Infinities and NaN where fp32 arithmetic has them, the rest within its rounding."""
    got, ref = got.cpu(), ref.cpu()
    assert torch.equal(got.isnan(), ref.isnan()), what
    assert torch.equal(got.isinf(), ref.isinf()), what
    inf, fin = ref.isinf(), ref.isfinite()
    assert torch.equal(got[inf], ref[inf]), what
    assert ((got[fin].double() - ref[fin].double()).norm() / ref[fin].double().norm()).item() < 1e-5, what


# (64, 64, 64) runs the fp32 kernel, the others the split kernel in every product
@pytest.mark.parametrize("M,K,N", [(64, 64, 64), (3000, 100, 1130), (130, 700, 1001), (730, 700, 1001)])
def test_infinities_and_nan(M, K, N):
    """Infinite, NaN and huge operands: the outputs they reach are those of fp32 arithmetic, the
    others are unharmed (their tile is formed again by fp32 MFMAs, so their rounding may change)."""
    from triton_tagi_amd.layers import Linear

    gen = torch.Generator("cuda").manual_seed(M + N)
    torch.manual_seed(M)
    for op in OPS:
        assert linear_plan(op, M, K, N).split_kernel == (M != 64), op
    layer = Linear(K, N, device="cuda")
    ma, Sa = inputs((M, K), gen)
    ma[1, 3], Sa[5, K - 1], ma[M - 1, 0], ma[7, 2] = float("inf"), float("nan"), 3e38, -3.4e38
    a, S, w, V = ma.cpu(), Sa.cpu(), layer.mw.cpu(), layer.Sw.cpu()
    mz, Sz = layer.forward(ma, Sa)
    m0, S0 = layer.forward(ma, None)
    same_specials(mz, a @ w + layer.mb.cpu(), "mz")
    same_specials(Sz, (a * a) @ V + S @ (w * w + V) + layer.Sb.cpu(), "Sz")
    same_specials(m0, a @ w + layer.mb.cpu(), "mz of a fixed input")
    same_specials(S0, (a * a) @ V + layer.Sb.cpu(), "Sz of a fixed input")
    # backward: one delta of each kind, and an activation that makes one row of the parameter
    # deltas infinite
    ma, Sa = inputs((M, K), gen)
    dm, dS = inputs((M, N), gen)
    ma[M - 1, K - 2], dm[3, 1], dS[9, N - 1], dm[M // 2, N // 2] = float("-inf"), float("inf"), float("nan"), 1e37
    layer.forward(ma, Sa)
    d_ma, d_Sa = layer.backward(dm, dS)
    a, d, e = ma.cpu(), dm.cpu(), dS.cpu()
    same_specials(d_ma, d @ w.T, "d_ma")
    same_specials(d_Sa, e @ (w * w).T, "d_Sa")
    same_specials(layer.delta_mw, V * (a.T @ d), "delta_mw")
    same_specials(layer.delta_Sw, V * V * ((a * a).T @ e), "delta_Sw")
    same_specials(layer.delta_mb, layer.Sb.cpu() * d.sum(0, keepdim=True), "delta_mb")
    same_specials(layer.delta_Sb, layer.Sb.cpu() ** 2 * e.sum(0, keepdim=True), "delta_Sb")


@pytest.mark.parametrize("C,Cout", [(64, 64), (42, 70)])
def test_infinities_and_nan_in_convolutions(C, Cout):
    from triton_tagi_amd.layers import Conv2D

    gen = torch.Generator("cuda").manual_seed(C)
    torch.manual_seed(C)
    B, H = 40, 14
    layer = Conv2D(C, Cout, 3, padding=1, device="cuda")
    for op in OPS:
        assert conv_plan(op, layer, B, H).split_kernel, op
    ma, Sa = inputs((B, C, H, H), gen)
    ma[0, 0, 0, 0], Sa[3, C - 1, 5, 6], ma[B - 1, 2, H - 1, H - 1] = float("inf"), float("nan"), -3e38
    mz, Sz = layer.forward(ma, Sa)
    W, V = layer.mw.cpu(), layer.Sw.cpu()
    patches = lambda t: F.unfold(t.cpu(), 3, padding=1).transpose(1, 2)  # noqa: E731
    image = lambda t: t.transpose(1, 2).reshape(B, Cout, H, H)  # noqa: E731
    p, q = patches(ma), patches(Sa)
    same_specials(mz, image(p @ W + layer.mb.cpu()), "mz")
    same_specials(Sz, image((p * p) @ V + q @ (W * W + V) + layer.Sb.cpu()), "Sz")
    ma, Sa = inputs((B, C, H, H), gen)
    dm, dS = inputs((B, Cout, H, H), gen)
    ma[5, 1, 2, 3], dm[0, 0, 4, 4], dS[7, Cout - 1, 0, 0] = float("inf"), float("-inf"), float("nan")
    layer.forward(ma, Sa)
    d_ma, d_Sa = layer.backward(dm, dS)
    rows = lambda t: t.cpu().reshape(B, Cout, H * H).transpose(1, 2)  # noqa: E731
    fold = lambda t: F.fold(t.transpose(1, 2), (H, H), 3, padding=1)  # noqa: E731
    d, e, p = rows(dm), rows(dS), patches(ma).reshape(-1, C * 9)
    same_specials(d_ma, fold(d @ W.T), "d_ma")
    same_specials(d_Sa, fold(e @ (W * W).T), "d_Sa")
    d, e = d.reshape(-1, Cout), e.reshape(-1, Cout)
    # fp32 arithmetic over the padding zeros of a patch: 0 times an infinite delta is NaN
    same_specials(layer.delta_mw, V * (p.T @ d), "delta_mw")
    same_specials(layer.delta_Sw, V * V * ((p * p).T @ e), "delta_Sw")


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
