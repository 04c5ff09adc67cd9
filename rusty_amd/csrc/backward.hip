// Input gradient through a frozen quantized Linear (LoRA fine-tuning):
//
//   dX[m, k_in] = dY[m, n_out] . deq(W)[n_out, k_in]
//
// the `grad_a = matmul_bt(grad, b)` step of MatMulNode::backward
// (rusty-autograd/src/lib.rs:152-158) with b the load-time-dequantized f32
// weight in [in, out] layout (rusty-graph/src/lib.rs:69-70): since
// b[i, o] = deq(W)[o, i], matmul_bt(grad, b) = dY . deq(W) in the stored
// [out, in] orientation, so W is read as it lies, with no transpose.  The
// weight gradient is not formed (the weight is frozen).
//
// One f32 accumulator per output updated by fma in ascending n_out (the f32
// matmul family's order).  The weight tile is dequantized while it is staged
// -- per-row codes f32(q) * s[row] (one rounding), affine codes
// (f32(u) * s[g]) + b[g] (two roundings, no contraction), exactly the values
// rq_qweight_dequantize writes -- so dX is bit-identical to the f32 matmul on
// the dequantized weight without that weight ever existing in memory.
// Memory: 1 B per weight element instead of 4.
//
// k_dx_chain runs on the f32 matrix cores (mfma_chain.hpp) and serves every
// call whose codes come in words (dx_chain_ok); k_qmatmul_dx, on the VALU,
// the rest (k_in or n_out not a multiple of 4, unaligned operands, groups that
// do not divide k_in) and short reductions into many outputs (dx_short).  Bound by the matrix instructions, which share the SIMD
// with the dequantization (3-4 VALU instructions per element of a tile, for
// 64 or 128 rows' products): us, VALU -> matrix cores, 512x4096x4096 affine 518 -> 140,
// per-row 372 -> 139; 2048x4096x4096 affine 1616 -> 587; 16 rows x 11008x4096
// 1144 -> 78 (the VALU kernel's 64x64 tiles left most CUs idle).
//
// k_qmatmul_dx: 64x64 output tiles per 256-thread block, 4x4 outputs per
// thread, steps of 32 along n_out; the next step's dY and code pieces are
// loaded into registers (8 codes and 8 dY values per thread) before the
// current step's fmas run.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "mfma_chain.hpp"

namespace rq {
namespace {

constexpr int BM = 64, BN = 64, BK = 32, TH = 256;

// The dequantized value of code c with its row's (per-row codes) or group's
// (affine) scale s and bias b.
template <int FMT>
__device__ __forceinline__ float deq1(uint32_t c, float s, float b) {
    if constexpr (FMT == RQ_Q_ROWWISE_I8) {
        return (float)(int8_t)c * s;
    } else {
        float v;
        {
#pragma clang fp contract(off)
            v = (float)c * s;
            v = v + b;
        }
        return v;
    }
}

// VW: codes 8-byte aligned and k_in % 8 == 0 (8 codes per load).
template <int FMT, bool DYF16, bool DXF16, bool VW>
__global__ __launch_bounds__(TH) void k_qmatmul_dx(const uint8_t *__restrict__ codes, const float *__restrict__ scales,
                                                   const float *__restrict__ biases, int group,
                                                   const void *__restrict__ dyv, void *__restrict__ dxv, int64_t m,
                                                   int64_t n_out, int64_t k_in) {
    __shared__ float As[BK][BM + 1];  // dY^T tile: [n_out step][row of dX]
    __shared__ float Bs[BK][BN + 4];  // deq(W) tile: [n_out step][column of dX]
    const int t = threadIdx.x;
    const int tx = t % 16, ty = t / 16;
    const int64_t m0 = (int64_t)blockIdx.y * BM, c0 = (int64_t)blockIdx.x * BN;
    // this thread's staging pieces: dY row ar, entries ac..ac+7 of the step
    // (contiguous along n_out); weight row br of the step, columns bc..bc+7
    const int ar = t / 4, ac = (t % 4) * 8;
    const int br = t / 8, bc = (t % 8) * 8;

    // raw loads (an out-of-range element loads element 0 of its operand) and
    // the zeroing of out-of-range elements at staging: a branch or a select
    // right after each load made the compiler wait for it before the fmas
    // raw loads into registers (conversions wait for their loads, so they are
    // done when staging): dY values as stored, 8 codes as one 8-byte word (or
    // 8 bytes where codes are unaligned or k_in % 8 != 0), their scales
    typedef _Float16 yt_t;
    std::conditional_t<DYF16, yt_t, float> yr[8];
    uint2 wq;        // VW
    uint8_t wb8[8];  // !VW
    float ws[FMT == RQ_Q_ROWWISE_I8 ? 1 : 8], wb[FMT == RQ_Q_ROWWISE_I8 ? 1 : 8];  // scales (and biases)
    auto load = [&](int64_t k0) {
        const int64_t gr = m0 + ar;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t gc = k0 + ac + e;
            const int64_t o = gr < m && gc < n_out ? gr * n_out + gc : 0;
            if constexpr (DYF16) yr[e] = static_cast<const _Float16 *>(dyv)[o];
            else yr[e] = static_cast<const float *>(dyv)[o];
        }
        const int64_t row = k0 + br, col = c0 + bc;
        if constexpr (VW) {  // k_in % 8 == 0: a thread's 8 columns are all in the row or all past it
            wq = *reinterpret_cast<const uint2 *>(codes + (row < n_out && col < k_in ? row * k_in + col : 0));
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) wb8[e] = codes[row < n_out && col + e < k_in ? row * k_in + col + e : 0];
        }
        if constexpr (FMT == RQ_Q_ROWWISE_I8) {
            ws[0] = scales[row < n_out ? row : 0];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t g = row < n_out && col + e < k_in ? (row * k_in + col + e) / group : 0;
                ws[e] = scales[g];
                wb[e] = biases ? biases[g] : 0.0f;
            }
        }
    };
    auto stage = [&](int64_t k0) {
        const int64_t gr = m0 + ar;
#pragma unroll
        for (int e = 0; e < 8; ++e) As[ac + e][ar] = gr < m && k0 + ac + e < n_out ? (float)yr[e] : 0.0f;
        const int64_t row = k0 + br, col = c0 + bc;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            uint32_t c;
            if constexpr (VW) c = ((e < 4 ? wq.x : wq.y) >> (8 * (e % 4))) & 0xFFu;
            else c = wb8[e];
            Bs[br][bc + e] = row < n_out && col + e < k_in
                                 ? deq1<FMT>(c, ws[FMT == RQ_Q_ROWWISE_I8 ? 0 : e], wb[FMT == RQ_Q_ROWWISE_I8 ? 0 : e])
                                 : 0.0f;
        }
    };

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;

    if (n_out > 0) load(0);
    for (int64_t k0 = 0; k0 < n_out; k0 += BK) {
        stage(k0);
        __syncthreads();
        if (k0 + BK < n_out) load(k0 + BK);  // in flight while this step's fmas run
        // the LDS values of step kk + 2 are requested before step kk's fmas
        // (three register sets, the loop fully unrolled)
        float av[3][4], bv[3][4];
        auto rd = [&](int st, int kk) {
#pragma unroll
            for (int i = 0; i < 4; ++i) av[st][i] = As[kk][ty + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[st][j] = Bs[kk][tx + 16 * j];
        };
        rd(0, 0);
        rd(1, 1);
#pragma unroll
        for (int kk = 0; kk < BK; ++kk) {
            if (kk + 2 < BK) rd((kk + 2) % 3, kk + 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(av[kk % 3][i], bv[kk % 3][j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t r = m0 + ty + 16 * i, c = c0 + tx + 16 * j;
            if (r < m && c < k_in) {
                if constexpr (DXF16) static_cast<_Float16 *>(dxv)[r * k_in + c] = (_Float16)acc[i][j];
                else static_cast<float *>(dxv)[r * k_in + c] = acc[i][j];
            }
        }
}

// ---- the same product on the f32 matrix cores (mfma_chain.hpp) ----------------
//
// deq(W) as the chain product's B panel, rows along the outputs (k_in) and
// the reduction over n_out: the codes of a piece (4 columns of one weight row)
// are loaded as one word with the row's scale, or with the scale and bias of
// the group the four columns share, and dequantized when the piece is staged,
// to the bits rq_qweight_dequantize writes.  Served: codes 4-byte aligned with
// k_in % 4 == 0, affine groups of a multiple of 4 dividing k_in (a group then
// holds whole pieces, and row r's groups start at r k_in / group).
template <int FMT, int R, int KC, int MF, int TILES, int TH_>
struct PanelW : PanelOLds<R, KC, MF, TILES, TH_> {
    using L = PanelOLds<R, KC, MF, TILES, TH_>;
    static constexpr bool AFFINE = FMT == RQ_Q_AFFINE_U8;
    struct Raw {
        uint32_t c[L::NP];
        float s[L::NP], b[AFFINE ? L::NP : 1];
    };
    struct Span {
        ChainSpan c, s, b;
    };
    const uint8_t *codes;  // column c0 of row 0
    const float *scales, *biases;
    int64_t ld, left;  // codes per row; columns from c0 on
    int gpr, group, c0;  // affine: groups per row; the panel's first column
    __device__ __forceinline__ uint32_t code_records(int rows) const {
        return rows > 0 ? (uint32_t)((rows - 1) * ld + left) : 0u;
    }
    __device__ __forceinline__ uint32_t scale_records(int rows) const {
        return (uint32_t)(AFFINE ? rows * gpr : rows) * 4u;
    }
    __device__ __forceinline__ Span first(int64_t k) const {
        const int rows = (int)(k < KC ? k : KC);
        Span sp{{reinterpret_cast<uint64_t>(codes), code_records(rows)},
                {reinterpret_cast<uint64_t>(scales), scale_records(rows)},
                {reinterpret_cast<uint64_t>(biases), biases ? scale_records(rows) : 0u}};
        return sp;
    }
    __device__ __forceinline__ void next(Span &sp, int st, int stages, int live) const {
        sp.c.base += KC * ld;
        sp.s.base += (AFFINE ? KC * (int64_t)gpr : KC) * 4;
        if constexpr (AFFINE) sp.b.base += KC * (int64_t)gpr * 4;
        if (st >= stages - 1) {
            const int rows = st == stages - 1 ? live : 0;
            sp.c.records = code_records(rows);
            sp.s.records = scale_records(rows);
            if constexpr (AFFINE) sp.b.records = biases ? scale_records(rows) : 0u;
        }
    }
    struct Off {  // a lane's byte offsets of the pieces' codes and scales
        uint32_t c[L::NP], s[L::NP];
    };
    __device__ __forceinline__ Off offsets(int t) const {
        Off o;
        const int col = c0 + 4 * (t % L::PR);
#pragma unroll
        for (int i = 0; i < L::NP; ++i) {
            const int r = t / L::PR + L::STEP * i;
            o.c[i] = (uint32_t)(r * ld + 4 * (t % L::PR));
            o.s[i] = (uint32_t)(AFFINE ? r * gpr + col / group : r) * 4u;
        }
        return o;
    }
    __device__ __forceinline__ void load(Raw &raw, int i, const Span &sp, const Off &o) const {
        raw.c[i] = __builtin_amdgcn_raw_buffer_load_b32(sp.c.rsrc(), o.c[i], 0, 0);
        raw.s[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sp.s.rsrc(), o.s[i], 0, 0));
        if constexpr (AFFINE)
            raw.b[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sp.b.rsrc(), o.s[i], 0, 0));
    }
    __device__ __forceinline__ void stage(const Raw &raw, int i, float *lds, int t) const {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = deq1<FMT>((raw.c[i] >> (8 * e)) & 0xFFu, raw.s[i], raw.b[AFFINE ? i : 0]);
        *reinterpret_cast<float4 *>(L::at(lds, i, t)) = make_float4(v[0], v[1], v[2], v[3]);
    }
};

template <int FMT, typename TY, int MF, int WM, int WN, int T, int KC, int MINB>
__global__ __launch_bounds__(TH, MINB) void k_dx_chain(const uint8_t *__restrict__ codes,
                                                       const float *__restrict__ scales,
                                                       const float *__restrict__ biases, int group,
                                                       const TY *__restrict__ dy, void *__restrict__ dx, bool dxf16,
                                                       int64_t m, int64_t n_out, int64_t k_in, uint32_t rows, uint32_t cols) {
    constexpr int TM = WM * T * MF, TN = WN * T * MF;
    using PA = PanelK<TY, true, TM, KC, MF, T, TH>;
    using PB = PanelW<FMT, TN, KC, MF, T, TH>;
    using Tile = ChainTile<PA, PB, MF, WM, WN, T, T, KC, 1>;
    __shared__ __attribute__((aligned(16))) float lds[Tile::LDS_FLOATS];
    uint32_t tr, tc;
    chain_tile_of(blockIdx.x, rows, cols, tr, tc);
    const int64_t m0 = (int64_t)tr * TM, c0 = (int64_t)tc * TN;
    PA pa;
    pa.p = dy + m0 * n_out;
    pa.ld = n_out;
    pa.left = m - m0;
    PB pb;
    pb.codes = codes + c0;
    pb.scales = scales;
    pb.biases = biases;
    pb.ld = k_in;
    pb.left = k_in - c0;
    pb.group = FMT == RQ_Q_AFFINE_U8 ? group : 1;
    pb.gpr = FMT == RQ_Q_AFFINE_U8 ? (int)(k_in / group) : 0;
    pb.c0 = (int)c0;
    typename Tile::acc_t acc[T][T];
    Tile::run(pa, pb, lds, n_out, threadIdx.x, acc);
    Tile::each(acc, threadIdx.x, [&](int r, int c, float v) {
        if (m0 + r < m && c0 + c < k_in) {
            const int64_t o = (m0 + r) * k_in + c0 + c;
            if (dxf16) static_cast<_Float16 *>(dx)[o] = (_Float16)v;
            else static_cast<float *>(dx)[o] = v;
        }
    });
}

bool dx_chain_ok(const rq_qweight &w, const void *dy, rq_dtype dyt, int64_t m, int num_cus) {
    const int64_t lim = (int64_t)1 << 29;
    if (!(aligned(w.codes, 4) && aligned(dy, dyt == RQ_F16 ? 8 : 16) && w.k_in % 4 == 0 && w.n_out % 4 == 0 &&
          w.k_in * 64 < lim && w.n_out * 128 < lim &&
          (w.format == RQ_Q_ROWWISE_I8 || (w.group % 4 == 0 && w.k_in % w.group == 0))))
        return false;
    const ChainTiles t = chain_tiles(m, w.k_in, w.n_out, num_cus);
    return grid_ok(t.rows * t.cols, TH);
}

// A gradient of one step of the VALU kernel (32 of n_out) is its output's
// write and a tile's fixed cost, of which that kernel, with more blocks in
// flight, has less: it serves such calls from the output counts below on (f32
// dY and dX, us, matrix cores -> VALU kernel, per-row, then affine: 512x4096
// outputs, n_out 4 6.8 -> 6.2, 7.0 -> 7.3; 28 6.5 -> 6.1, 7.0 -> 7.6; 1024x4096,
// 28 10.9 -> 9.6, 11.5 -> 11.0; 4096x4096, 4 29.0 -> 22.4, 30.8 -> 24.8; 28 29.0 ->
// 24.0, 30.7 -> 28.0; 32 27.6 -> 25.9, 28.7 -> 31.1, at k_in % 8 = 4 17.3 -> 18.9;
// from 36 on the matrix cores: 2048x4096 20.9 against 23.4).
bool dx_short(const rq_qweight &w, int64_t m) {
    if (cdiv(m, BM) > 65535) return false;  // the VALU kernel's grid
    const bool rowwise = w.format == RQ_Q_ROWWISE_I8;
    auto from = [&](int log2) { return m * w.k_in >= ((int64_t)1 << log2); };
    return w.n_out <= (rowwise && from(23) && w.k_in % 8 == 0 ? 32 : from(rowwise ? 21 : 22) ? 28 : 0);
}

template <int FMT, bool DYF16>
int launch_fmt(const rq_qweight &w, const void *dy, void *dx, bool dxf16, int64_t m, dim3 grid, hipStream_t s) {
    const uint8_t *codes = static_cast<const uint8_t *>(w.codes);
    const bool vw = w.k_in % 8 == 0 && aligned(codes, 8);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(TH), 0, s, codes, w.scales, w.biases, w.group, dy, dx, m, w.n_out,
                           w.k_in);
    };
    if (dxf16) vw ? go(k_qmatmul_dx<FMT, DYF16, true, true>) : go(k_qmatmul_dx<FMT, DYF16, true, false>);
    else vw ? go(k_qmatmul_dx<FMT, DYF16, false, true>) : go(k_qmatmul_dx<FMT, DYF16, false, false>);
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

template <int FMT, typename TY>
int launch_chain(const rq_qweight &w, const void *dyv, void *dx, bool dxf16, int64_t m, int num_cus, hipStream_t s) {
    const ChainTiles t = chain_tiles(m, w.k_in, w.n_out, num_cus);
    const dim3 grid((unsigned)(t.rows * t.cols));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(TH), 0, s, static_cast<const uint8_t *>(w.codes), w.scales, w.biases,
                           w.group, static_cast<const TY *>(dyv), dx, dxf16, m, w.n_out, w.k_in, (uint32_t)t.rows,
                           (uint32_t)t.cols);
    };
    switch (t.shape) {
    case CHAIN_128: go(k_dx_chain<FMT, TY, 32, 2, 2, 2, 32, 1>); break;
    case CHAIN_64: go(k_dx_chain<FMT, TY, 32, 2, 2, 1, 32, 2>); break;
    case CHAIN_32: go(k_dx_chain<FMT, TY, 16, 2, 2, 1, 64, 1>); break;
    case CHAIN_16x64: go(k_dx_chain<FMT, TY, 16, 1, 4, 1, 64, 1>); break;
    case CHAIN_64x16: go(k_dx_chain<FMT, TY, 16, 4, 1, 1, 64, 1>); break;
    }
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

}  // namespace

int launch_qmatmul_dx(const rq_qweight &w, const void *dy, rq_dtype dyt, void *dx, rq_dtype dxt, int64_t m,
                      int num_cus, hipStream_t s) {
    const bool dyf16 = dyt == RQ_F16, dxf16 = dxt == RQ_F16;
    if (dx_chain_ok(w, dy, dyt, m, num_cus) && !dx_short(w, m)) {
        if (w.format == RQ_Q_ROWWISE_I8)
            return dyf16 ? launch_chain<RQ_Q_ROWWISE_I8, _Float16>(w, dy, dx, dxf16, m, num_cus, s)
                         : launch_chain<RQ_Q_ROWWISE_I8, float>(w, dy, dx, dxf16, m, num_cus, s);
        return dyf16 ? launch_chain<RQ_Q_AFFINE_U8, _Float16>(w, dy, dx, dxf16, m, num_cus, s)
                     : launch_chain<RQ_Q_AFFINE_U8, float>(w, dy, dx, dxf16, m, num_cus, s);
    }
    const int64_t gx = cdiv(w.k_in, BN), gy = cdiv(m, BM);
    if (gx > 0x7fffffff || gy > 65535)
        return fail(RQ_ERR_SHAPE, "input-gradient grid too large (m=%lld k_in=%lld)", (long long)m,
                    (long long)w.k_in);
    const dim3 grid((unsigned)gx, (unsigned)gy);
    if (w.format == RQ_Q_ROWWISE_I8)
        return dyf16 ? launch_fmt<RQ_Q_ROWWISE_I8, true>(w, dy, dx, dxf16, m, grid, s)
                     : launch_fmt<RQ_Q_ROWWISE_I8, false>(w, dy, dx, dxf16, m, grid, s);
    return dyf16 ? launch_fmt<RQ_Q_AFFINE_U8, true>(w, dy, dx, dxf16, m, grid, s)
                 : launch_fmt<RQ_Q_AFFINE_U8, false>(w, dy, dx, dxf16, m, grid, s);
}

}  // namespace rq

// ---- Input gradient on the matrix cores (per-row int8 codes) ----
//
// dX[m][k] = sum_n dY[m][n] s[n] q[n][k] is a GEMM whose reduction runs along
// n_out, while the int8 rows of W are contiguous along k_in: the matrix cores
// need the reduction contiguous in each lane's operand.  So a table built once
// per weight (load time, rq_qweight_dx_table) holds the codes transposed and
// written twice side by side, qt[k][j] = q[j mod n][k] for j < 2 n_out, and
// k_in unit scales; each dY row becomes v = dY s (f32, one rounding) scaled by
// the power of two 2^-e that puts max |v| in [2^14, 2^15), then two fp16
// halves x2[m] = [fp16(v 2^-e) | fp16(v 2^-e - hi)] (hi + lo = v 2^-e to
// ~2^-22 relative).  The prefill GEMM (gemm.hip) then computes
// dX[m][k] = 2^e sum_j x2[m][j] qt[k][j]: exact fp16 x int8 products, f32
// sums -- the f32 bar against the exact product, not the chain's bit pattern
// (rq_qmatmul_dx keeps that).  Memory: the table is 2 B per weight element.
namespace rq {
namespace {

constexpr int TT = 64;  // transpose tile, bytes per side

// qt[k][j] = qt[k][j + n] = q[j][k], one 64 x 64 tile per block; n % 16 == 0,
// k % 16 == 0, so every 16-byte piece lies wholly inside or outside.
__global__ __launch_bounds__(256) void k_dx_transpose(const uint8_t *__restrict__ q, uint8_t *__restrict__ qt,
                                                      int64_t n, int64_t k) {
    __shared__ uint8_t tile[TT][TT + 4];  // [n local][k local]
    const int t = threadIdx.x, r = t / 4, c = (t % 4) * 16;
    const int64_t n0 = (int64_t)blockIdx.y * TT, k0 = (int64_t)blockIdx.x * TT;
    {
        const int64_t gn = n0 + r, gk = k0 + c;
        const uint4 v = gn < n && gk < k ? *reinterpret_cast<const uint4 *>(q + gn * k + gk) : make_uint4(0, 0, 0, 0);
        const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 16; ++e) tile[r][c + e] = (uint8_t)(wd[e / 4] >> (8 * (e % 4)));
    }
    __syncthreads();
    const int64_t gk = k0 + r, gn = n0 + c;  // row gk of qt, its bytes gn .. gn + 15
    if (gk < k && gn < n) {
        uint32_t wd[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 16; ++e) wd[e / 4] |= (uint32_t)tile[c + e][r] << (8 * (e % 4));
        const uint4 v = make_uint4(wd[0], wd[1], wd[2], wd[3]);
        *reinterpret_cast<uint4 *>(qt + gk * 2 * n + gn) = v;
        *reinterpret_cast<uint4 *>(qt + gk * 2 * n + n + gn) = v;
    }
}

__global__ __launch_bounds__(256) void k_fill_ones(float *__restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 1.0f;
}

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

// Row i of dY (one block): v[j] = dY[i][j] s[j]; the row maximum (DPP steps
// and one barrier), 2^e with max |v| 2^-e in [2^14, 2^15) (e >= -126: 2^e
// stays a normal f32; a zero row gives e = 0), then x2[i][j] = hi,
// x2[i][n + j] = lo and xs[i] = 2^e.  Pieces of 8 values (n % 8 == 0): with
// VEC (dY and s 16-byte aligned) 16- or 32-byte loads, and with NI > 0
// (n <= 2048 NI) each thread keeps its NI pieces in registers from the
// maximum to the split, so the row is read once; otherwise it is read twice
// (the second time from L2).
template <bool DYF16, bool VEC, int NI>
__global__ __launch_bounds__(256) void k_dx_split(const void *__restrict__ dy, const float *__restrict__ s,
                                                  _Float16 *__restrict__ x2, float *__restrict__ xs, int64_t n) {
    __shared__ float wmax[4];
    const int64_t row = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63;
    const int n8 = (int)(n / 8);
    auto piece = [&](int i, float *v) {  // v = dY[row][8i + e] * s[8i + e]
        float sv[8], dv[8];
        if constexpr (VEC) {
            const float4 s0 = reinterpret_cast<const float4 *>(s)[2 * i], s1 = reinterpret_cast<const float4 *>(s)[2 * i + 1];
            sv[0] = s0.x; sv[1] = s0.y; sv[2] = s0.z; sv[3] = s0.w; sv[4] = s1.x; sv[5] = s1.y; sv[6] = s1.z; sv[7] = s1.w;
            if constexpr (DYF16) {
                const half8_t h = reinterpret_cast<const half8_t *>(static_cast<const _Float16 *>(dy) + row * n)[i];
#pragma unroll
                for (int e = 0; e < 8; ++e) dv[e] = (float)h[e];
            } else {
                const float4 *d4 = reinterpret_cast<const float4 *>(static_cast<const float *>(dy) + row * n);
                const float4 a = d4[2 * i], b = d4[2 * i + 1];
                dv[0] = a.x; dv[1] = a.y; dv[2] = a.z; dv[3] = a.w; dv[4] = b.x; dv[5] = b.y; dv[6] = b.z; dv[7] = b.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t j = (int64_t)8 * i + e;
                sv[e] = s[j];
                dv[e] = DYF16 ? (float)static_cast<const _Float16 *>(dy)[row * n + j]
                              : static_cast<const float *>(dy)[row * n + j];
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = dv[e] * sv[e];
    };
    auto amax8 = [](const float *v) {
        float a = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) a = fmaxf(a, fabsf(v[e]));
        return a;
    };
    float amax = 0.0f;
    float held[NI > 0 ? NI : 1][8];
    if constexpr (NI > 0) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {  // every load in flight before the first use
            const int i = t + 256 * j;
            if (i < n8) piece(i, held[j]);
            else
#pragma unroll
                for (int e = 0; e < 8; ++e) held[j][e] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) amax = fmaxf(amax, amax8(held[j]));
    } else {
        for (int i = t; i < n8; i += 256) {
            float v[8];
            piece(i, v);
            amax = fmaxf(amax, amax8(v));
        }
    }
    amax = fmaxf(amax, dppf<0xB1>(amax));   // quad_perm [1,0,3,2]
    amax = fmaxf(amax, dppf<0x4E>(amax));   // quad_perm [2,3,0,1]
    amax = fmaxf(amax, dppf<0x141>(amax));  // row_half_mirror
    amax = fmaxf(amax, dppf<0x140>(amax));  // row_mirror: each 16-lane row holds its maximum
    const auto rl = [](float v, int l) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
    };
    amax = fmaxf(fmaxf(rl(amax, 0), rl(amax, 16)), fmaxf(rl(amax, 32), rl(amax, 48)));
    if (lane == 0) wmax[t >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int e = max(__builtin_amdgcn_frexp_expf(amax) - 15, -126);
    half8_t *hr = reinterpret_cast<half8_t *>(x2 + row * 2 * n);
    auto split = [&](int i, const float *v) {
        half8_t hi, lo;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float w = __builtin_amdgcn_ldexpf(v[q], -e);
            hi[q] = (_Float16)w;
            lo[q] = (_Float16)(w - (float)hi[q]);
        }
        hr[i] = hi;
        hr[n8 + i] = lo;
    };
    if constexpr (NI > 0) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            const int i = t + 256 * j;
            if (i < n8) split(i, held[j]);
        }
    } else {
        for (int i = t; i < n8; i += 256) {
            float v[8];
            piece(i, v);
            split(i, v);
        }
    }
    if (t == 0) xs[row] = __builtin_amdgcn_ldexpf(1.0f, e);
}

bool dx_table_ok(const rq_qweight &w) {
    return w.format == RQ_Q_ROWWISE_I8 && w.n_out >= 32 && w.n_out % 32 == 0 && w.k_in >= 16 && w.k_in % 16 == 0 &&
           2 * w.n_out <= (1 << 21) && w.k_in <= 0x7fffffff && aligned(w.codes, 16);
}
size_t dx_codes_bytes(const rq_qweight &w) { return ((size_t)2 * w.n_out * w.k_in + 255) & ~size_t(255); }

}  // namespace
}  // namespace rq

using namespace rq;

extern "C" {

size_t rq_qweight_dx_table_bytes(const rq_qweight *w) {
    if (!w || check_qweight(w) != RQ_OK || !dx_table_ok(*w)) return 0;
    return dx_codes_bytes(*w) + (size_t)w->k_in * 4;
}

int rq_qweight_dx_table(rq_ctx *ctx, const rq_qweight *w, void *table, size_t table_bytes, rq_stream stream) {
    RQ_ENTER(ctx);
    int st = check_qweight(w);
    if (st != RQ_OK) return st;
    if (!dx_table_ok(*w))
        return fail(RQ_ERR_UNSUPPORTED, "the matrix-core input gradient takes per-row int8 codes, 16-byte aligned, "
                                        "n_out a multiple of 32, k_in a multiple of 16");
    const size_t need = rq_qweight_dx_table_bytes(w);
    if (!table || table_bytes < need || !aligned(table, 256))
        return fail(RQ_ERR_INVALID_ARGUMENT, "table of %zu bytes (256-byte aligned), %zu needed", table_bytes, need);
    hipStream_t s = pick(ctx, stream);
    const int64_t n = w->n_out, k = w->k_in;
    if (cdiv(k, TT) > 0x7fffffff || cdiv(n, TT) > 65535) return fail(RQ_ERR_SHAPE, "weight too large to transpose");
    uint8_t *qt = static_cast<uint8_t *>(table);
    hipLaunchKernelGGL(k_dx_transpose, dim3((unsigned)cdiv(k, TT), (unsigned)cdiv(n, TT)), dim3(256), 0, s,
                       static_cast<const uint8_t *>(w->codes), qt, n, k);
    RQ_LAUNCH_CHECK();
    float *ones = reinterpret_cast<float *>(qt + dx_codes_bytes(*w));
    hipLaunchKernelGGL(k_fill_ones, dim3((unsigned)std::min<int64_t>(cdiv(k, 256), 4096)), dim3(256), 0, s, ones, k);
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

size_t rq_qmatmul_dx_mfma_workspace(int64_t m, int64_t n_out) {
    if (m < 0 || n_out < 0) return 0;
    return (((size_t)m * (size_t)n_out * 4 + 255) & ~size_t(255)) + (size_t)m * 4;
}

int rq_qmatmul_dx_mfma(rq_ctx *ctx, const rq_qweight *w, const void *table, const void *dy, rq_dtype dy_dtype,
                       void *dx, rq_dtype dx_dtype, int64_t m, void *workspace, size_t workspace_bytes,
                       rq_stream stream) {
    RQ_ENTER(ctx);
    int st = check_qweight(w);
    if (st != RQ_OK) return st;
    if ((dy_dtype != RQ_F16 && dy_dtype != RQ_F32) || (dx_dtype != RQ_F16 && dx_dtype != RQ_F32))
        return fail(RQ_ERR_INVALID_ARGUMENT, "dtype must be RQ_F16 or RQ_F32");
    if (!dx_table_ok(*w))
        return fail(RQ_ERR_UNSUPPORTED, "the matrix-core input gradient takes per-row int8 codes, 16-byte aligned, "
                                        "n_out a multiple of 32, k_in a multiple of 16");
    if (m < 0) return fail(RQ_ERR_SHAPE, "negative m");
    int64_t t;
    if (!mul_ok(m, w->k_in, &t) || !mul_ok(m, 2 * w->n_out, &t) || m > 0x7fffffff)
        return fail(RQ_ERR_SHAPE, "shape overflows");
    if (m == 0) return RQ_OK;
    if (!dx || !dy || !table) return fail(RQ_ERR_INVALID_ARGUMENT, "null gradient or table pointer");
    if (!aligned(table, 256)) return fail(RQ_ERR_INVALID_ARGUMENT, "table must be 256-byte aligned");
    const size_t need = rq_qmatmul_dx_mfma_workspace(m, w->n_out);
    if (!workspace || workspace_bytes < need || !aligned(workspace, 256))
        return fail(RQ_ERR_INVALID_ARGUMENT, "workspace of %zu bytes (256-byte aligned), %zu needed",
                    workspace_bytes, need);
    hipStream_t s = pick(ctx, stream);
    const int64_t n = w->n_out, k = w->k_in;
    _Float16 *x2 = static_cast<_Float16 *>(workspace);
    float *xs = reinterpret_cast<float *>(static_cast<char *>(workspace) + (((size_t)m * n * 4 + 255) & ~size_t(255)));
    {
        const bool vec = aligned(dy, 16) && aligned(w->scales, 16);
        const int64_t per = cdiv(n / 8, 256);  // 8-value pieces per thread
        auto go = [&](auto f16, auto v, auto ni) {
            hipLaunchKernelGGL((k_dx_split<decltype(f16)::value, decltype(v)::value, decltype(ni)::value>),
                               dim3((unsigned)m), dim3(256), 0, s, dy, w->scales, x2, xs, n);
        };
        auto by_ni = [&](auto f16, auto v) {
            if (per <= 1) go(f16, v, std::integral_constant<int, 1>{});
            else if (per <= 2) go(f16, v, std::integral_constant<int, 2>{});
            else if (per <= 4) go(f16, v, std::integral_constant<int, 4>{});
            else go(f16, v, std::integral_constant<int, 0>{});
        };
        auto by_vec = [&](auto f16) {
            if (vec) by_ni(f16, std::true_type{});
            else by_ni(f16, std::false_type{});
        };
        if (dy_dtype == RQ_F16) by_vec(std::true_type{});
        else by_vec(std::false_type{});
        RQ_LAUNCH_CHECK();
    }
    // the transposed problem: k_in rows of 2 n_out codes, unit scales
    const uint8_t *qt = static_cast<const uint8_t *>(table);
    const rq_qweight wt{qt, reinterpret_cast<const float *>(qt + dx_codes_bytes(*w)), nullptr, k, 2 * n,
                        RQ_Q_ROWWISE_I8, 0, nullptr};
    st = launch_gemm_f16_scaled(wt, wt.scales, x2, xs, dx, dx_dtype, m, ctx->num_cus, gemm_workspace(ctx, s), s);
    if (st == RQ_ERR_UNSUPPORTED) return fail(st, "dx pointer alignment (8 bytes fp16, 16 bytes f32) not met");
    return st;
}

}  // extern "C"

// For the tests, no part of the C ABI: the tile (bm * 1000 + bn) of the
// matrix-core kernel that serves an input gradient in f32 with aligned
// operands, 0 for the VALU kernel.  Host arithmetic.
extern "C" int rusty_dx_kernel(int fmt, int group, int64_t m, int64_t n_out, int64_t k_in, int num_cus) {
    using namespace rq;
    rq_qweight w{};
    w.format = fmt;
    w.group = group;
    w.n_out = n_out;
    w.k_in = k_in;
    if (!dx_chain_ok(w, nullptr, RQ_F32, m, num_cus) || dx_short(w, m)) return 0;
    return chain_tile_id(chain_tiles(m, k_in, n_out, num_cus));
}
