// The f32 matmul family on the f32 matrix cores (mfma_chain.hpp).  One
// translation unit per variant (matmul_ab.hip, matmul_abt.hip, matmul_atb.hip)
// instantiates launch_mfma; matmul_f32.hip chooses the kernel of a call.
#pragma once

#include <type_traits>

#include "mfma_chain.hpp"

namespace rq {

int launch_mfma_ab(const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus, hipStream_t s);
int launch_mfma_ab_f16(const _Float16 *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus, hipStream_t s);
int launch_mfma_abt(const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus, hipStream_t s);
int launch_mfma_atb(const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus, hipStream_t s);

// Operands that load in whole pieces of four elements.
template <typename TA>
bool vec_a(int v, const TA *a, int64_t m, int64_t k) {
    return aligned(a, 4 * sizeof(TA)) && (v == MM_ATB ? m : k) % 4 == 0;
}
inline bool vec_b(int v, const float *b, int64_t k, int64_t n) { return aligned(b, 16) && (v == MM_ABT ? k : n) % 4 == 0; }

namespace {

constexpr int MTH = 256;  // threads per block

// Bound by the f32 matrix instructions: 4096^3 978 us, 140 TFLOP/s of the 154
// they reach from registers (the vendor's f32 GEMM of the same shape: 1008 us);
// the VALU kernel, at one fma per lane and cycle, took 2270.  Below a full
// grid of 64x64 tiles the chain of each output bounds it (3.3 ns per k).
// TA: float, or _Float16 for an fp16 A (MM_AB).  VA, VB: operands that load in
// whole 16-byte pieces; a ragged row pitch costs little (537x2773x2853 93 us,
// element loads along the rows).
template <int V, typename TA, bool VA, bool VB, int MF, int WM, int WN, int T, int KC, int MINB>
__global__ __launch_bounds__(MTH, MINB) void k_matmul_mfma(const TA *__restrict__ a, const float *__restrict__ b,
                                                          float *__restrict__ out, int64_t m, int64_t k, int64_t n,
                                                          uint32_t rows, uint32_t cols) {
    constexpr int TM_ = WM * T * MF, TN_ = WN * T * MF;
    static_assert(V != MM_ATB || std::is_same_v<TA, float>, "fp16 A: C = A.B only");
    using PA = std::conditional_t<V == MM_ATB, PanelO<VA, TM_, KC, MF, T, MTH>, PanelK<TA, VA, TM_, KC, MF, T, MTH>>;
    using PB = std::conditional_t<V == MM_ABT, PanelK<float, VB, TN_, KC, MF, T, MTH>, PanelO<VB, TN_, KC, MF, T, MTH>>;
    using Tile = ChainTile<PA, PB, MF, WM, WN, T, T, KC, 1>;
    __shared__ __attribute__((aligned(16))) float lds[Tile::LDS_FLOATS];
    uint32_t tr, tc;
    chain_tile_of(blockIdx.x, rows, cols, tr, tc);
    const int64_t m0 = (int64_t)tr * TM_, n0 = (int64_t)tc * TN_;
    PA pa;
    PB pb;
    if constexpr (V == MM_ATB) {
        pa.p = a + m0;
        pa.ld = m;
    } else {
        pa.p = a + m0 * k;
        pa.ld = k;
    }
    pa.left = m - m0;
    pb.p = V == MM_ABT ? b + n0 * k : b + n0;
    pb.ld = V == MM_ABT ? k : n;
    pb.left = n - n0;
    typename Tile::acc_t acc[T][T];
    Tile::run(pa, pb, lds, k, threadIdx.x, acc);
    Tile::each(acc, threadIdx.x, [&](int r, int c, float v) {
        if (m0 + r < m && n0 + c < n) out[(m0 + r) * n + n0 + c] = v;
    });
}

template <int V, typename TA, bool VA, bool VB>
int launch_mfma_vec(const TA *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus,
                    hipStream_t s) {
    const ChainTiles t = chain_tiles(m, n, k, num_cus);
    const dim3 grid((unsigned)(t.rows * t.cols));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(MTH), 0, s, a, b, out, m, k, n, (uint32_t)t.rows, (uint32_t)t.cols);
    };
    switch (t.shape) {
    case CHAIN_128: go(k_matmul_mfma<V, TA, VA, VB, 32, 2, 2, 2, 32, 1>); break;
    case CHAIN_64: go(k_matmul_mfma<V, TA, VA, VB, 32, 2, 2, 1, 32, 2>); break;
    case CHAIN_32: go(k_matmul_mfma<V, TA, VA, VB, 16, 2, 2, 1, 64, 1>); break;
    case CHAIN_16x64: go(k_matmul_mfma<V, TA, VA, VB, 16, 1, 4, 1, 64, 1>); break;
    case CHAIN_64x16: go(k_matmul_mfma<V, TA, VA, VB, 16, 4, 1, 1, 64, 1>); break;
    }
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

template <int V, typename TA>
int launch_mfma(const TA *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus, hipStream_t s) {
    const bool va = vec_a(V, a, m, k), vb = vec_b(V, b, k, n);
    if (va && vb) return launch_mfma_vec<V, TA, true, true>(a, b, out, m, k, n, num_cus, s);
    if constexpr (V != MM_ABT && std::is_same_v<TA, float>) {  // (A . B^T: both follow k)
        if (va) return launch_mfma_vec<V, TA, true, false>(a, b, out, m, k, n, num_cus, s);
        if (vb) return launch_mfma_vec<V, TA, false, true>(a, b, out, m, k, n, num_cus, s);
    }
    return launch_mfma_vec<V, TA, false, false>(a, b, out, m, k, n, num_cus, s);
}

}  // namespace
}  // namespace rq
