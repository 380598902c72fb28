"""The planner's launches cover their products at every size (host only, no kernel runs)."""

import ctypes
import itertools

from triton_tagi_amd import _lib

SCRATCH_BYTES = 128 << 20  # the fixed scratch of tagi_linear_fwd_noalloc
OPS = (_lib.OP_FWD, _lib.OP_FWD_FIXED, _lib.OP_BWD_DELTA, _lib.OP_WGRAD)


def linear_plan(op, M, K, N, ws=-1):
    p = _lib.Plan()
    _lib.call("tagi_linear_plan", op, M, K, N, ws, ctypes.byref(p))
    return p


def conv_plan(op, g, ws=-1):
    p = _lib.Plan()
    _lib.call("tagi_conv2d_plan", op, ctypes.byref(g), ws, ctypes.byref(p))
    return p


def geom(B, C, H, Cout, k, s):
    Ho = (H + 2 * (k // 2) - k) // s + 1
    return _lib.ConvGeom(B, C, H, H, Cout, k, s, k // 2, k // 2, Ho, Ho)


def covers(p, R, C, K):
    assert p.splits >= 1 and p.k_chunk >= 1 and p.tile_rows >= 16 and p.tile_cols >= 16
    assert p.tiles_rows * p.tile_rows >= R > (p.tiles_rows - 1) * p.tile_rows
    assert p.tiles_cols * p.tile_cols >= C > (p.tiles_cols - 1) * p.tile_cols
    assert p.splits * p.k_chunk >= K > (p.splits - 1) * p.k_chunk
    assert p.splits == 1 or p.k_chunk % (32 if p.split_kernel else 16) == 0


def test_linear_plans_cover_their_products():
    sizes = (1, 3, 10, 64, 257, 1000, 2048, 4096, 4097, 5120, 11008, 50257)
    for M, K, N in itertools.product(sizes, repeat=3):
        if max(M * K, (K + 1) * N, M * N) >= 1 << 31:
            continue
        for op in OPS:
            R, C, red = {_lib.OP_BWD_DELTA: (M, K, N), _lib.OP_WGRAD: (K + 1, N, M)}.get(op, (M, N, K))
            full, none = linear_plan(op, M, K, N), linear_plan(op, M, K, N, 0)
            covers(full, R, C, red)
            covers(none, R, C, red)
            assert none.splits == 1
            need = 8 * R * C * full.splits if full.splits > 1 else 0
            name = ("tagi_linear_fwd_ws_bytes", "tagi_linear_fwd_ws_bytes", "tagi_linear_bwd_delta_ws_bytes",
                    "tagi_linear_wgrad_ws_bytes")[op]
            assert getattr(_lib.load(), name)(M, K, N) >= need


def test_linear_forward_above_the_fixed_scratch():
    """Outputs whose one pair of partial planes is larger than the scratch run unsplit where
    the scratch's rule leaves no split, and are never refused."""
    for M, K, N in ((4097, 4096, 4097), (4096, 5120, 5120), (5000, 4096, 4096), (10000, 2048, 2048),
                    (2048, 5120, 13824), (512, 2048, 50257), (4096, 2880, 4608), (1600, 4096, 11008)):
        assert 8 * M * N > SCRATCH_BYTES
        p = linear_plan(_lib.OP_FWD, M, K, N)
        covers(p, M, N, K)
        assert p.splits == 1 and _lib.load().tagi_linear_fwd_ws_bytes(M, K, N) <= 16 * 8 * M * N


def test_conv_plans_cover_their_products():
    for B, C, H, Cout, k, s in itertools.product((1, 7, 128), (1, 3, 42, 64, 512), (4, 15, 32), (4, 10, 70, 512),
                                                 (1, 3, 5), (1, 2)):
        if k > H:
            continue
        Ho = (H + 2 * (k // 2) - k) // s + 1
        g = geom(B, C, H, Cout, k, s)
        taps = max(-(-(k - a) // s) for a in range(min(s, k)))
        for op in OPS:
            R, cols, red = {_lib.OP_BWD_DELTA: (B * (-(-H // s)) ** 2, C, taps * taps * Cout),
                            _lib.OP_WGRAD: (C * k * k + 1, Cout, B * Ho * Ho)}.get(op, (B * Ho * Ho, Cout, C * k * k))
            covers(conv_plan(op, g), R, cols, red)
            none = conv_plan(op, g, 0)
            covers(none, R, cols, red)
            assert none.splits == 1


def test_products_that_stay_with_the_fp32_kernel():
    """One product beyond each line of the choice between the kernels, and one before it."""
    F, F0, D, W = OPS
    linear = [  # op, fp32 kernel, split kernel
        (W, (3, 4096, 11008), (4, 4096, 11008)), (W, (1, 4096, 11008), (8, 4096, 11008)),  # too few terms
        (F, (256, 784, 256), (512, 784, 256)), (F, (1024, 64, 256), (2048, 64, 256)),  # small products
        (F, (65536, 256, 3), (65536, 256, 4)), (D, (65536, 3, 256), (65536, 4, 256)),  # narrow sides
    ]
    for op, a, b in linear:
        assert linear_plan(op, *a).split_kernel == 0, (op, a)
        assert linear_plan(op, *b).split_kernel == 1, (op, b)
    conv = [
        (F, (128, 3, 32, 64, 3, 1), (128, 5, 32, 64, 3, 1)),  # element-wise patches under one k tile
        (D, (50, 66, 27, 70, 3, 1), (50, 62, 27, 70, 3, 1)),  # and their input deltas of many channels
        (D, (200, 64, 64, 3, 3, 2), (200, 64, 64, 4, 3, 2)),  # a stride phase of too few terms
    ]
    for op, a, b in conv:
        for ws in (-1, 0):
            assert conv_plan(op, geom(*a), ws).split_kernel == 0, (op, a)
            assert conv_plan(op, geom(*b), ws).split_kernel == 1, (op, b)


def test_tiles_left_out():
    """Beside loaders of any alignment and of element-wise patches, and of short reductions."""
    F, F0, D, W = OPS
    big = [(256, 128), (256, 64)]
    rows = (4, 60, 115, 437, 1111, 4097, 16385, 60000)
    for M, K, N in itertools.product(rows, (24, 100, 129, 515, 2001, 7157), (16, 120, 129, 1023, 2001, 11008)):
        for op, out, short, red in ((F, [(256, 128)], 128, K), (F0, [(256, 128), (128, 128)], 64, K),
                                    (D, [(128, 128)], 0, N), (W, [(128, 128)], 256, M)):
            p = linear_plan(op, M, K, N)
            tile = (p.tile_cols, p.tile_rows) if op == W else (p.tile_rows, p.tile_cols)
            bad = out if N % 4 or (op != D and K % 4) else []
            bad = bad + (big if red < (256 if op == W else 128) else [])
            bad = bad + ([(128, 128), (128, 64)] if red < short else [])
            assert not p.split_kernel or tile not in bad, (op, M, K, N)
    for B, C, H, Cout, k in itertools.product((8, 100), (6, 42, 63), (14, 32), (10, 70, 255), (1, 3, 5)):
        for op, out in ((F, [(128, 64), (128, 32)]), (F0, [(128, 128)]), (D, [(128, 32), (128, 128), (256, 128)])):
            if op == D and Cout % 4 == 0:
                continue
            p = conv_plan(op, geom(B, C, H, Cout, k, 1))
            assert not p.split_kernel or (p.tile_rows, p.tile_cols) not in out, (op, B, C, H, Cout, k)
