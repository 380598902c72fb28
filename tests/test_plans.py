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
        g = _lib.ConvGeom(B, C, H, H, Cout, k, s, k // 2, k // 2, Ho, Ho)
        taps = max(-(-(k - a) // s) for a in range(min(s, k)))
        for op in OPS:
            R, cols, red = {_lib.OP_BWD_DELTA: (B * (-(-H // s)) ** 2, C, taps * taps * Cout),
                            _lib.OP_WGRAD: (C * k * k + 1, Cout, B * Ho * Ho)}.get(op, (B * Ho * Ho, Cout, C * k * k))
            covers(conv_plan(op, g), R, cols, red)
            none = conv_plan(op, g, 0)
            covers(none, R, cols, red)
            assert none.splits == 1
