"""The library's dispatch rules, evaluated on the host (no kernel runs): which
tile or kernel a call takes on a device of 256 CUs."""
import ctypes

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


def matmul_kernel(variant, m, k, n):
    """0 tiled, 1 register-staged chains, 2 ring chains, else the matrix-core tile (rows, columns)."""
    i32, i64 = ctypes.c_int, ctypes.c_int64
    t = _fn("rusty_matmul_kernel", i32, i64, i64, i64, i32)(variant, m, k, n, CUS)
    return t if t < 1000 else divmod(t, 1000)


def dx_kernel(fmt, group, m, n_out, k_in):
    """0 for the VALU kernel, else the matrix-core tile (rows, columns)."""
    i32, i64 = ctypes.c_int, ctypes.c_int64
    t = _fn("rusty_dx_kernel", i32, i32, i64, i64, i64, i32)(fmt, group, m, n_out, k_in, CUS)
    return t if t < 1000 else divmod(t, 1000)
