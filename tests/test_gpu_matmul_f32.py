"""GPU parity of the f32 matmul family against the oracle, bit-exact.

rq_matmul    <- kernels.wgsl:7-54    (matmul_tiled)  / lib.rs:4403-4453
rq_matmul_bt <- kernels.wgsl:234-242 (matmul_bt)     / lib.rs:4299-4349
rq_matmul_at <- kernels.wgsl:244-252 (matmul_at)     / lib.rs:4351-4401

The device keeps one f32 accumulator per output updated in ascending k with
fma, so it must equal the oracle's fused k-ascending loop bit for bit.
"""
import numpy as np
import pytest

from oracle import oracle as orc
from rusty_amd import UnifiedTensor
from tile_query import matmul_kernel

pytestmark = pytest.mark.gpu

# Products of a few k-steps take the 64x64 tiled kernel, A.B^T with few outputs
# the ring chains, one 16x16 tile of outputs the register-staged chains, the
# rest the matrix cores: k past a chunk and not a multiple of 32, k = 0, every
# column-tile width.  All must match the oracle bit for bit.
SHAPES = [(2, 2, 2), (1, 1024, 1024), (8, 1024, 1024), (65, 33, 70), (128, 256, 96), (3, 0, 5), (1, 4096, 4096),
          (1, 4097, 16), (5, 1000, 40), (33, 600, 9), (7, 300, 3), (2, 513, 100), (512, 4096, 16),
          (512, 200, 520), (1030, 64, 600),
          # 16-byte rows with ragged row and column blocks and a partial last chunk
          (20, 520, 44), (12, 700, 36),
          # 9 to 16 columns over whole k-chunks, rows no multiple of 4
          (17, 1024, 9), (101, 1536, 16)]


def _run(engine, ctx, op, a, b, m, n):
    A, B = UnifiedTensor.new(ctx, a), UnifiedTensor.new(ctx, b)
    out = UnifiedTensor.new(ctx, np.full((m, n), np.nan, np.float32))
    getattr(engine, op)(ctx, A, B, out)
    return out.to_vec()


def test_identity_known_answer(ctx, engine):
    # rusty-backend/examples/ops_test.rs:13-17
    got = _run(engine, ctx, "matmul", np.array([[1, 2], [3, 4]], np.float32), np.eye(2, dtype=np.float32), 2, 2)
    assert got.ravel().tolist() == [1, 2, 3, 4]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_matmul_family_bit_exact(ctx, engine, m, k, n):
    g = np.random.default_rng(m * 7 + k + n)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    want = orc.matmul(a, b, fused=True)
    assert np.array_equal(_run(engine, ctx, "matmul", a, b, m, n).view(np.uint32), want.view(np.uint32))
    bt = np.ascontiguousarray(b.T)
    assert np.array_equal(_run(engine, ctx, "matmul_bt", a, bt, m, n).view(np.uint32),
                          orc.matmul_bt(a, bt, fused=True).view(np.uint32))
    at = np.ascontiguousarray(a.T)
    assert np.array_equal(_run(engine, ctx, "matmul_at", at, b, m, n).view(np.uint32),
                          orc.matmul_at(at, b, fused=True).view(np.uint32))


def test_k_ascending_order(ctx, engine):
    a = np.array([[1e8, 1.0, -1e8, 1.0]], np.float32)
    assert _run(engine, ctx, "matmul", a, np.ones((4, 1), np.float32), 1, 1).item() == 1.0


def test_shape_mismatch_raises(ctx, engine):
    A = UnifiedTensor.new(ctx, np.zeros((2, 3), np.float32))
    B = UnifiedTensor.new(ctx, np.zeros((4, 5), np.float32))
    out = UnifiedTensor.empty(ctx, [2, 5])
    with pytest.raises(ValueError):
        engine.matmul(ctx, A, B, out)


# The matrix-core kernel on its 32x32 and 64x64 tiles: outputs one short of, at
# and past whole tiles, k below a stage (32 or 64), at whole stages and one past,
# row pitches in whole 16-byte pieces and not (every tile over many stages: below).
MFMA_SHAPES = [(2050, 52, 2052), (1920, 64, 2047), (1023, 33, 1025), (1000, 96, 1000), (255, 100, 255),
               (97, 65, 130), (64, 128, 64), (63, 127, 65), (15, 70, 1500), (16, 64, 4100), (1500, 70, 15),
               (2100, 129, 16), (33, 17, 31), (17, 18, 19), (1, 20, 300), (300, 21, 1)]


@pytest.mark.parametrize("m,k,n", MFMA_SHAPES)
def test_matrix_core_tiles_bit_exact(ctx, engine, m, k, n):
    test_matmul_family_bit_exact(ctx, engine, m, k, n)


# Every tile over more than seven stages (the ring of three turns twice, registers refill) and a
# partial last one, ragged in rows and columns; operands in whole 16-byte pieces and by element.
LONG_SHAPES = [((16, 64), 8, 460, 11008), ((16, 64), 9, 461, 11009), ((64, 16), 11008, 460, 8),
               ((64, 16), 11009, 461, 9), ((32, 32), 100, 460, 1100), ((32, 32), 101, 461, 1099),
               ((64, 64), 40, 460, 11008), ((64, 64), 41, 461, 11009), ((128, 128), 2500, 460, 1300),
               ((128, 128), 2501, 461, 1301)]


@pytest.mark.parametrize("tile,m,k,n", LONG_SHAPES)
def test_matrix_core_long_reductions_bit_exact(ctx, engine, tile, m, k, n):
    assert [matmul_kernel(v, m, k, n) for v in range(3)] == [tile] * 3
    test_matmul_family_bit_exact(ctx, engine, m, k, n)


@pytest.mark.parametrize("k", [17, 30, 65])
def test_padding_and_specials(ctx, engine, k):
    """A partial last stage leaves every accumulator as it is: a sum that
    underflowed to -0 keeps its sign, infinities and NaN stay in their rows
    and columns, subnormals are kept."""
    m, n = 70, 66
    g = np.random.default_rng(k)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)
    a[3], b[:, 5] = -1e-30, 1e-30  # outputs (3, 5): the products underflow to -0
    a[7], b[:, 9] = 1e-42, np.float32(0.75)  # subnormal operands
    a[11, 2], b[4, 13] = np.inf, np.nan
    with np.errstate(all="ignore"):
        want = orc.matmul(a, b, fused=True)
        for op, x, y in (("matmul", a, b), ("matmul_bt", a, np.ascontiguousarray(b.T)),
                         ("matmul_at", np.ascontiguousarray(a.T), b)):
            got = _run(engine, ctx, op, x, y, m, n)
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(got), nan)
            assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])
    assert np.signbit(want[3, 5]) and want[3, 5] == 0


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_unaligned_operands(ctx, engine, shift):
    """Operands that start at any float (a view into a larger buffer)."""
    m, k, n = 130, 72, 68
    g = np.random.default_rng(shift)
    a = g.standard_normal((m, k), dtype=np.float32)
    b = g.standard_normal((k, n), dtype=np.float32)

    def at(x):
        t = UnifiedTensor.new(ctx, np.concatenate([np.zeros(shift, np.float32), x.ravel()]))
        v = UnifiedTensor(ctx, t.ptr + 4 * shift, x.shape, t.dtype, owner=False)
        v._base = t
        return v

    out = UnifiedTensor.empty(ctx, [m, n])
    for op, x, y in (("matmul", a, b), ("matmul_bt", a, np.ascontiguousarray(b.T)),
                     ("matmul_at", np.ascontiguousarray(a.T), b)):
        getattr(engine, op)(ctx, at(x), at(y), out)
        assert np.array_equal(out.to_vec().view(np.uint32), orc.matmul(a, b, fused=True).view(np.uint32))
