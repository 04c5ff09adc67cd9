"""CPU checks of the kernels' dispatch rules: host arithmetic of the library,
evaluated for a 256-CU device.  No kernel runs here."""
import pytest

from tile_query import dx_kernel, gemm_tile, matmul_kernel


def _threads(t, m, n, per_block):
    return -(-m // t[0]) * -(-n // t[1]) * per_block


@pytest.mark.parametrize("big", [1 << 27, (1 << 29) - 8, 1 << 29, (1 << 29) + 40, 1 << 30])
@pytest.mark.parametrize("small", [1, 8, 17, 32, 64, 100])
def test_grids_stay_below_the_launch_limit(big, small):
    """A launch has fewer than 2^32 threads along x: no rule moves a product
    whose larger tiles fit that to smaller ones that do not."""
    for m, n in ((small, big), (big, small)):
        for variant in range(3):
            for k in (56, 260):
                t = matmul_kernel(variant, m, k, n)
                assert isinstance(t, int) or _threads(t, m, n, 256) < 1 << 32, (variant, m, k, n, t)
        for fmt, group in ((0, 0), (1, 4)):
            t = dx_kernel(fmt, group, m, 64, n & ~3)
            assert isinstance(t, int) or _threads(t, m, n & ~3, 256) < 1 << 32, (fmt, m, n, t)
            for width in (64, 128, 200, 256):
                t = gemm_tile(fmt, min(big, (1 << 29) + 40), width, 64)
                assert _threads(t, min(big, (1 << 29) + 40), width, 512 if t[1] >= 128 else 256) < 1 << 32, (width, t)


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


def test_short_reductions_take_smaller_tiles():
    """A round of 128x128 tiles has a fixed cost (its outputs' write) that a
    short reduction does not hide: 64x64 there, 128x128 for long ones."""
    for k in (64, 128, 256):
        assert all(matmul_kernel(v, 2048, k, 4096) == (64, 64) for v in range(3))
        assert dx_kernel(0, 0, 2048, k, 4096) == dx_kernel(1, 64, 2048, k, 4096) == (64, 64)
    for k in (64, 128, 256):
        assert matmul_kernel(0, 700, k, 3000) == (64, 64)
    assert matmul_kernel(0, 2048, 512, 2048) == matmul_kernel(0, 4096, 4096, 4096) == (128, 128)
    assert matmul_kernel(0, 512, 4096, 16) == (32, 32)


@pytest.mark.parametrize("fmt,group,rows", [(0, 0, 512), (1, 64, 1024)])
def test_short_input_gradients_of_many_outputs(fmt, group, rows):
    """One step of the VALU kernel into many outputs is its; anything longer or
    smaller, and more rows than its grid takes, the matrix cores'."""
    for m in (rows, 2 * rows, 8192):
        for n_out in (4, 16, 28):
            assert dx_kernel(fmt, group, m, n_out, 4096) == 0
        assert dx_kernel(fmt, group, m, 36, 4096) != 0
    assert dx_kernel(fmt, group, rows - 64, 28, 4096) != 0
    assert (dx_kernel(fmt, group, 2048, 32, 4096) == 0) == (fmt == 0)
    assert dx_kernel(fmt, group and 4, 2048, 32, 4100) != 0
    assert dx_kernel(fmt, group, 512, 256, 4096) != 0
    assert dx_kernel(fmt, group, 65535 * 64 + 1, 16, 256) != 0


def test_gemm_tile_outside_the_fitted_times():
    """What the fitted times miss: one round of 128x256 tiles over a short K
    stays, three 64x64 tiles per CU need a clear gain; measured the other way
    round, both lost."""
    for m, n, k in ((554, 10904, 320), (1179, 4672, 384), (922, 6579, 320)):
        assert gemm_tile(0, m, n, k) == (128, 256)
    assert gemm_tile(0, 1453, 6816, 384) == (64, 128)  # more than a round: 23.3 us on 128x256, 18.4
    assert gemm_tile(0, 1066, 2720, 1152) == (128, 128)
    assert gemm_tile(0, 157, 8448, 896) == (64, 64)  # 128x64 17.3 us, 64x64 8.5
    assert gemm_tile(1, 390, 4992, 1408) == (64, 64)


def test_thin_products_that_load_by_element():
    """9 to 16 columns over whole k-chunks with rows that are no multiple of 4
    stay on the register-staged chains; ragged k and whole pieces do not."""
    for variant, m, n in ((0, 17, 9), (0, 100, 9), (2, 17, 9), (2, 17, 16), (2, 101, 16)):
        for k in (512, 1024, 4096):
            assert matmul_kernel(variant, m, k, n) == 1
        assert matmul_kernel(variant, m, 1022, n) == (32, 32) or variant == 2 and matmul_kernel(variant, m, 1022, n) != 1
    assert matmul_kernel(2, 2001, 1024, 16) == 1 and matmul_kernel(2, 2001, 4096, 16) != 1
    for variant, m, n in ((0, 100, 16), (2, 100, 16), (2, 500, 16), (0, 101, 16)):  # whole pieces
        assert matmul_kernel(variant, m, 4096, n) not in (0, 1, 2)
    assert matmul_kernel(2, 17, 4096, 8) != 1 and matmul_kernel(2, 17, 4096, 17) != 1
