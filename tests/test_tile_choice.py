"""CPU checks of the kernels' dispatch rules: host arithmetic of the library,
evaluated for a 256-CU device.  No kernel runs here."""
import ctypes

import pytest

from rusty_amd import _lib

CUS = 256


def _fn(name, *argtypes):
    f = getattr(_lib.lib(), name)
    f.argtypes, f.restype = list(argtypes), ctypes.c_int
    return f


def gemm_tile(fmt, m, n_out, k_in, pair=False):
    """(rows, columns) of the prefill GEMM's tile, None where gate and up are two products."""
    i32, i64 = ctypes.c_int, ctypes.c_int64
    t = _fn("rusty_gemm_tile", i32, i64, i64, i64, i32, i32)(fmt, m, n_out, k_in, CUS, int(pair))
    return None if t < 0 else divmod(t, 1000)


@pytest.mark.parametrize("fmt", [0, 1])
def test_pair_tile_rows_stay_below_the_mask_offset(fmt):
    """The fused gate/up copy-out masks pieces with byte offset 2^31: no tile's
    rows of h (2 bytes per value) may reach it, whatever the width."""
    edges = [(1 << 31) // (2 * bm) for bm in (192, 128)]  # 5592405 and 8388608
    widths = [e // 8 * 8 + d for e in edges for d in (-8, 0, 8)] + [6_000_008, 7_000_024, 8_388_600, 16_777_208]
    served = 0
    for inter in widths:
        for m in (64, 128, 192, 300, 384, 576, 1024, 2048):
            for k in (64, 1024, 4096):
                t = gemm_tile(fmt, m, inter, k, pair=True)
                if t is not None:
                    served += 1
                    assert t[0] * inter * 2 < 1 << 31, (m, inter, k, t)
    assert served > 50  # widths below 128-row tiles' limit are still one launch
