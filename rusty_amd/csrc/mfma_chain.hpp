// Tiled products on the f32 matrix cores with the bits of a k-ascending fma
// chain per output.
//
// v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 update every accumulator
// entry by one fused multiply-add per k of the instruction, in ascending k,
// rounding each to f32 (nearest even, subnormals kept): the result equals
//   for (k...) acc = fmaf(a[k], b[k], acc)
// bit for bit.  Compared on MI355X against that loop on the host for both
// shapes, 64 k-steps, 40960 outputs each: normal values, exponents spread over
// 2^-12..2^12 and 2^-40..2^40, subnormal inputs, products and sums, overflow
// to infinity and NaN -- no output differs.  So a kernel that walks k in order
// with one accumulator per output keeps the reference's order whatever its
// tiling.  From registers, in a bare loop, the two run at 154 and 139 TFLOP/s
// (the one-wide VALU fma of the same chain: 78.6 peak); one dependent chain
// advances 13.2 ns (32x32x2) and 3.3 ns (16x16x4) per k, the VALU's 3.2 ns.
//
// These instructions share the SIMD with the vector ALU: every VALU
// instruction between them costs its own cycles (a 128x128 tile's k-loop ran
// 4096^3 in 897 us with nothing but the matrix instructions, 919 with the LDS
// reads, 1003 with 12 VALU instructions per staged piece, 1223 with the
// address arithmetic of clamped 64-bit loads).  So the k-loop below has almost
// none: global loads are buffer loads at fixed per-lane offsets from a scalar
// base that advances by a stage (what lies past the operand reads as zero),
// pieces go to LDS as loaded, LDS addresses are per-lane constants plus
// immediates (the loop is unrolled over the LDS stages), and the padding of a
// partial last stage is written over the staged values once, at that stage.
//
// A block computes a (WM TM MF) x (WN TN MF) tile with WM x WN waves of
// TM x TN matrix-core tiles.  Operand panels pass through a ring of three LDS
// stages of KC k-steps; PF further stages are held in registers.  Lane l
// supplies k = KS s + l / MF of step s (KS = 2 or 4):
//  * an operand whose rows run along k (PanelK) is staged by rows, the 4 KS
//    k-steps of four matrix instructions as KS chunks of 16 bytes, chunk q
//    holding one lane half's (quarter's) values k % KS = q: one 16-byte read
//    gives a lane four steps (4-byte reads of rows in their stored order:
//    4096^3 A.B^T 1213 -> 1071 us).  Chunks are XOR-swizzled by row so that 16
//    rows of a tile hit all banks;
//  * an operand whose rows run along the outputs (PanelO) is staged
//    [k][output]; a lane's T tiles take T adjacent outputs (output T i + j of
//    the wave's share is entry i of tile j): one 4 T-byte read per step.
// Fragments of the next four steps are read while the current four multiply,
// across stages too (a stage is complete one barrier before it is needed).
#pragma once

#include "common.hpp"

namespace rq {

typedef unsigned chain_u32x4 __attribute__((ext_vector_type(4)));

template <int MF>
struct MfmaF32;
template <>
struct MfmaF32<32> {
    typedef float acc_t __attribute__((ext_vector_type(16)));
    static constexpr int KS = 2, NR = 16;
    static __device__ __forceinline__ acc_t mul(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    // row of the tile that entry r of lane l holds (its column is l % 32)
    static __device__ __forceinline__ int row(int r, int l) { return 8 * (r >> 2) + 4 * (l >> 5) + (r & 3); }
};
template <>
struct MfmaF32<16> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    static constexpr int KS = 4, NR = 4;
    static __device__ __forceinline__ acc_t mul(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int r, int l) { return 4 * (l >> 4) + r; }
};

// The part of an operand that one stage's loads may touch, kept in scalar
// registers: `base` moves on by a stage at a time and `records` (bytes) bounds
// it, so what lies past the panel's rows or past k reads as zero.
struct ChainSpan {
    uint64_t base;
    uint32_t records;
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc() const {
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((uint64_t)hi << 32 | lo), 0,
                                                 __builtin_amdgcn_readfirstlane(records), 0x00020000);
    }
};

// ---- operand panels -----------------------------------------------------------
// A panel is R outputs x KC k-steps of one operand, loaded by TH threads in
// NP pieces of 4 elements each.  load() fetches piece i of a stage, stage()
// writes it to LDS, pad() overwrites what of it lies at or past `live` k-steps:
// with -0 for one operand and +0 for the other, so that the padded steps add
// -0 and leave every accumulator as it is, -0 included.  Outputs past the
// operand's rows get whatever the loads return: they are never stored.

// Rows along k: element (output r, k) at p[r ld + k].  VEC: 16-byte aligned
// base and ld % 4 == 0 (fp16: 8-byte).  T: float or _Float16 (widened exactly).
template <typename T, bool VEC, int R, int KC, int MF, int TILES, int TH>
struct PanelK {
    static constexpr bool along_k = true;
    static constexpr int KS = MfmaF32<MF>::KS;
    static constexpr int NP = R * KC / 4 / TH, PR = KC / 4, STEP = TH / PR;
    static_assert(R * KC % (4 * TH) == 0 && TH % PR == 0 && KC <= 64 && KC >= 16, "panel");
    static constexpr int RPB = 64 / KC;  // rows per pass over the banks
    static_assert(STEP % (RPB * PR) == 0 && MF % (RPB * PR) == 0, "pieces and tiles share a row's swizzle");
    static constexpr int FLOATS = R * KC;
    static constexpr int NA = KC / (4 * KS);  // LDS read addresses per lane: one per group of four steps
    typedef T vec4 __attribute__((ext_vector_type(4)));
    struct Raw {
        vec4 v[NP];
    };
    const T *p;        // row r0 of the operand
    int64_t ld, left;  // rows from r0 on
    // the host keeps R ld below 2^29 (chain_tile_fits): offsets and records fit 31 bits
    __device__ __forceinline__ ChainSpan first(int64_t k) const {
        const int64_t r = left < R ? left : R;
        return {reinterpret_cast<uint64_t>(p), (uint32_t)(((r - 1) * ld + k) * (int64_t)sizeof(T))};
    }
    // moves on to stage st
    __device__ __forceinline__ void next(ChainSpan &s, int, int, int) const {
        s.base += KC * sizeof(T);
        s.records = (uint32_t)max((int)s.records - (int)(KC * sizeof(T)), 0);
    }
    static __device__ __forceinline__ int swz(int r) { return (r / RPB) % PR; }
    // Row and k (within the stage) of element e of piece i: with VEC a piece is
    // four k of a row; without, four rows at one k, so that the lanes of each
    // 4-byte load still read runs of a row.
    static __device__ __forceinline__ int row(int i, int e, int t) {
        return VEC ? t / PR + STEP * i : t / KC + TH / KC * (4 * i + e);
    }
    static __device__ __forceinline__ int kof(int e, int t) { return VEC ? 4 * (t % PR) + e : t % KC; }
    struct Off {  // a lane's byte offsets
        uint32_t v[VEC ? NP : 4 * NP];
    };
    __device__ __forceinline__ Off offsets(int t) const {
        Off o;
#pragma unroll
        for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int e = 0; e < (VEC ? 1 : 4); ++e)
                o.v[VEC ? i : 4 * i + e] = (uint32_t)(row(i, e, t) * ld + kof(e, t)) * (uint32_t)sizeof(T);
        return o;
    }
    __device__ __forceinline__ void load(Raw &raw, int i, const ChainSpan &s, const Off &o) const {
        const auto rs = s.rsrc();
        if constexpr (VEC && sizeof(T) == 4) {
            raw.v[i] = __builtin_bit_cast(vec4, __builtin_amdgcn_raw_buffer_load_b128(rs, o.v[i], 0, 0));
        } else if constexpr (VEC) {
            raw.v[i] = __builtin_bit_cast(vec4, __builtin_amdgcn_raw_buffer_load_b64(rs, o.v[i], 0, 0));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (sizeof(T) == 4)
                    raw.v[i][e] = __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, o.v[4 * i + e], 0, 0));
                else
                    raw.v[i][e] = __builtin_bit_cast(
                        T, (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, o.v[4 * i + e], 0, 0));
            }
        }
    }
    // LDS float index of element e of the thread's piece i
    static __device__ __forceinline__ int at(int i, int e, int t) {
        const int r = row(VEC ? 0 : i, e, t), k = kof(e, t), c = k / 4;
        return r * KC + 4 * ((c / KS * KS + k % KS) ^ swz(r)) + c % KS + k % 4 / KS * 2 + (VEC ? STEP * i * KC : 0);
    }
    __device__ __forceinline__ void stage(const Raw &raw, int i, float *lds, int t) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[at(i, e, t)] = (float)raw.v[i][e];
    }
    static __device__ __forceinline__ void pad(float *lds, int i, int live, int t, float v) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (kof(e, t) >= live) lds[at(i, e, t)] = v;
    }
    // LDS float index of the lane's chunk of group g, its wave's tile 0
    static __device__ __forceinline__ void addresses(int (&ad)[NA], int w, int lane) {
        const int r = w * TILES * MF + lane % MF;
#pragma unroll
        for (int g = 0; g < NA; ++g) ad[g] = r * KC + 4 * ((KS * g + lane / MF) ^ swz(r));
    }
    // the lane's values of steps 4g .. 4g + 3 of its tiles
    static __device__ __forceinline__ void fragment(float (&f)[TILES][4], const float *lds, const int (&ad)[NA], int g) {
#pragma unroll
        for (int j = 0; j < TILES; ++j) {
            const float4 v = *reinterpret_cast<const float4 *>(lds + ad[g] + j * MF * KC);
            f[j][0] = v.x;
            f[j][1] = KS == 2 ? v.z : v.y;
            f[j][2] = KS == 2 ? v.y : v.z;
            f[j][3] = v.w;
        }
    }
    // output (within the panel) of entry i of tile j of wave w
    static __device__ __forceinline__ int out(int w, int j, int i) { return (w * TILES + j) * MF + i; }
};

// Where the staged [k][output] rows put output c: XORed by 16 or 32 floats so
// that the KS rows a step reads lie on different banks (TILES MF floats each).
template <int R, int MF, int TILES>
__device__ __forceinline__ int swz_o(int k) {
    constexpr int W = MF * TILES;  // floats a wave reads of a row
    if constexpr (MF == 32) return W == 32 && R % 64 == 0 ? 32 * (k & 1) : 0;
    else if constexpr (W == 16) return R % 64 == 0 ? 16 * (k & 3) : (R == 32 ? 16 * ((k >> 1) & 1) : 0);
    else return W == 32 && R % 64 == 0 ? 32 * (k & 1) : 0;
}

// The [k][output] side shared by operands stored that way and by weights
// dequantized on the way.
template <int R, int KC, int MF, int TILES, int TH>
struct PanelOLds {
    static constexpr bool along_k = false;
    static constexpr int KS = MfmaF32<MF>::KS;
    static constexpr int NP = R * KC / 4 / TH, PR = R / 4, STEP = TH / PR;
    static_assert(R * KC % (4 * TH) == 0 && TH % PR == 0 && STEP % KS == 0 && R % 4 == 0, "panel");
    static constexpr int FLOATS = KC * R;
    static constexpr int NA = 1;
    static __device__ __forceinline__ float *at(float *lds, int i, int t) {
        const int k = t / PR;
        return lds + k * R + ((4 * (t % PR)) ^ swz_o<R, MF, TILES>(k)) + STEP * i * R;
    }
    static __device__ __forceinline__ void pad(float *lds, int i, int live, int t, float v) {
        if (t / PR + STEP * i >= live) *reinterpret_cast<float4 *>(at(lds, i, t)) = make_float4(v, v, v, v);
    }
    static __device__ __forceinline__ void addresses(int (&ad)[NA], int w, int lane) {
        const int q = lane / MF;
        ad[0] = q * R + ((w * TILES * MF + TILES * (lane % MF)) ^ swz_o<R, MF, TILES>(q));
    }
    static __device__ __forceinline__ void fragment(float (&f)[TILES][4], const float *lds, const int (&ad)[NA], int g) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float *o = lds + ad[0] + KS * (4 * g + s) * R;
            if constexpr (TILES == 1) {
                f[0][s] = *o;
            } else {
                static_assert(TILES == 2, "tiles per wave");
                const float2 v = *reinterpret_cast<const float2 *>(o);
                f[0][s] = v.x;
                f[1][s] = v.y;
            }
        }
    }
    static __device__ __forceinline__ int out(int w, int j, int i) { return w * TILES * MF + TILES * i + j; }
};

// Rows along the outputs: element (k, output c) at p[k ld + c].  VEC: 16-byte
// aligned base and ld % 4 == 0.
template <bool VEC, int R, int KC, int MF, int TILES, int TH>
struct PanelO : PanelOLds<R, KC, MF, TILES, TH> {
    using L = PanelOLds<R, KC, MF, TILES, TH>;
    struct Raw {
        float4 v[L::NP];
    };
    const float *p;    // output r0 of k-row 0
    int64_t ld, left;  // outputs from r0 on
    // the host keeps KC ld below 2^29 (chain_tile_fits)
    __device__ __forceinline__ uint32_t records(int rows) const {
        return rows > 0 ? (uint32_t)((rows - 1) * ld + left) * 4u : 0u;
    }
    __device__ __forceinline__ ChainSpan first(int64_t k) const {
        return {reinterpret_cast<uint64_t>(p), records((int)(k < KC ? k : KC))};
    }
    // moves on to stage st; the last one holds `live` k-steps
    __device__ __forceinline__ void next(ChainSpan &s, int st, int stages, int live) const {
        s.base += KC * ld * 4;
        if (st >= stages - 1) s.records = st == stages - 1 ? records(live) : 0u;
    }
    // Without VEC a piece is one output at four k-rows, so that the lanes of
    // each 4-byte load still read runs of a row.
    static_assert(VEC || TH % R == 0, "panel");
    static __device__ __forceinline__ int krow(int i, int e, int t) { return t / R + TH / R * (4 * i + e); }
    struct Off {
        uint32_t v[VEC ? L::NP : 4 * L::NP];
    };
    __device__ __forceinline__ Off offsets(int t) const {
        Off o;
#pragma unroll
        for (int i = 0; i < L::NP; ++i) {
            if constexpr (VEC) {
                o.v[i] = (uint32_t)((t / L::PR + L::STEP * i) * ld + 4 * (t % L::PR)) * 4u;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) o.v[4 * i + e] = (uint32_t)(krow(i, e, t) * ld + t % R) * 4u;
            }
        }
        return o;
    }
    __device__ __forceinline__ void load(Raw &raw, int i, const ChainSpan &s, const Off &o) const {
        const auto rs = s.rsrc();
        if constexpr (VEC) {
            raw.v[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, o.v[i], 0, 0));
        } else {
            float e[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                e[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o.v[4 * i + j], 0, 0));
            raw.v[i] = make_float4(e[0], e[1], e[2], e[3]);
        }
    }
    static __device__ __forceinline__ int at1(int i, int e, int t) {
        const int k = krow(i, e, t);
        return k * R + ((t % R) ^ swz_o<R, MF, TILES>(k));
    }
    __device__ __forceinline__ void stage(const Raw &raw, int i, float *lds, int t) const {
        if constexpr (VEC) {
            *reinterpret_cast<float4 *>(L::at(lds, i, t)) = raw.v[i];
        } else {
            lds[at1(i, 0, t)] = raw.v[i].x;
            lds[at1(i, 1, t)] = raw.v[i].y;
            lds[at1(i, 2, t)] = raw.v[i].z;
            lds[at1(i, 3, t)] = raw.v[i].w;
        }
    }
    static __device__ __forceinline__ void pad(float *lds, int i, int live, int t, float v) {
        if constexpr (VEC) {
            L::pad(lds, i, live, t, v);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (krow(i, e, t) >= live) lds[at1(i, e, t)] = v;
        }
    }
};

// ---- the product -----------------------------------------------------------------

template <class PA, class PB, int MF, int WM, int WN, int TM, int TN, int KC, int PF>
struct ChainTile {
    using M = MfmaF32<MF>;
    using acc_t = typename M::acc_t;
    static constexpr int KS = M::KS, TH = 64 * WM * WN;
    static constexpr int STAGE = PA::FLOATS + PB::FLOATS;
    static constexpr int GROUPS = KC / (4 * KS);  // four steps each
    static_assert(GROUPS % 2 == 0, "fragment sets alternate across stages");
    static constexpr int NP = PA::NP + PB::NP, NM = GROUPS * 4 * TM * TN;  // pieces and matrix instructions of a stage
    static constexpr int NS = 3;
    static constexpr int LDS_FLOATS = NS * STAGE;
    static constexpr int UNROLL = PF % NS == 0 ? PF : NS * PF;

    static __device__ __forceinline__ void run(const PA &a, const PB &b, float *lds, int64_t k, int t,
                                               acc_t (&acc)[TM][TN]) {
        const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), wm = w / WN, wn = w % WN;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < M::NR; ++r) acc[i][j][r] = 0.0f;
        if (k <= 0) return;
        typename PA::Raw ra[PF + 2];  // [PF], [PF + 1]: stages 0 and 1, before the loop only
        typename PB::Raw rb[PF + 2];
        const int stages = (int)((k + KC - 1) / KC);
        const int tail = k % KC ? stages - 1 : -1, live = (int)(k - (int64_t)(stages - 1) * KC);
        const auto oa = a.offsets(t);
        const auto ob = b.offsets(t);
        auto sa = a.first(k);
        auto sb = b.first(k);
        // loads run one stage after another: the spans move on behind a stage's last piece
        auto load = [&](int u, int i, int st) {
            if (i < PA::NP) a.load(ra[u], i, sa, oa);
            else b.load(rb[u], i - PA::NP, sb, ob);
            if (i == PA::NP - 1) a.next(sa, st + 1, stages, live);
            if (i == NP - 1) b.next(sb, st + 1, stages, live);
        };
        auto stage = [&](int u, int i, float *to) {
            if (i < PA::NP) a.stage(ra[u], i, to, t);
            else b.stage(rb[u], i - PA::NP, to + PA::FLOATS, t);
        };
        auto pad = [&](int st, float *to) {  // each thread over the pieces it staged itself
            if (st != tail) return;
#pragma unroll
            for (int i = 0; i < PA::NP; ++i) a.pad(to, i, live, t, -0.0f);
#pragma unroll
            for (int i = 0; i < PB::NP; ++i) b.pad(to + PA::FLOATS, i, live, t, 0.0f);
        };
        // stages 0 and 1 to LDS, 2 .. PF + 1 in registers, all requested at once
#pragma unroll
        for (int st = 0; st < PF + 2; ++st)
#pragma unroll
            for (int i = 0; i < NP; ++i) load(st < 2 ? PF + st : st - 2, i, st);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
#pragma unroll
            for (int i = 0; i < NP; ++i) stage(PF + st, i, lds + st * STAGE);
            pad(st, lds + st * STAGE);
        }
        __syncthreads();
        int aa[PA::NA], ab[PB::NA];
        PA::addresses(aa, wm, lane);
        PB::addresses(ab, wn, lane);
        float fa[2][TM][4], fb[2][TN][4];
        PA::fragment(fa[0], lds, aa, 0);
        PB::fragment(fb[0], lds + PA::FLOATS, ab, 0);
        for (int st = 0;;) {
#pragma unroll
            for (int u = 0; u < UNROLL; ++u) {
                const float *la = lds + (u % NS) * STAGE, *ln = lds + ((u + 1) % NS) * STAGE;
                float *to = lds + ((u + 2) % NS) * STAGE;  // last read in stage st - 1, before the previous barrier
#pragma unroll
                for (int g = 0; g < GROUPS; ++g) {
                    const float *lg = g + 1 < GROUPS ? la : ln;
                    PA::fragment(fa[(g + 1) & 1], lg, aa, (g + 1) % GROUPS);
                    PB::fragment(fb[(g + 1) & 1], lg + PA::FLOATS, ab, (g + 1) % GROUPS);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int s = 0; s < 4; ++s)
#pragma unroll
                        for (int i = 0; i < TM; ++i)
#pragma unroll
                            for (int j = 0; j < TN; ++j) {
                                acc[i][j] = M::mul(fa[g & 1][i][s], fb[g & 1][j][s], acc[i][j]);
                                const int n = ((g * 4 + s) * TM + i) * TN + j;
#pragma unroll
                                for (int c = 0; c < NP; ++c)
                                    if (c * NM / NP == n) {
                                        stage(u % PF, c, to);
                                        load(u % PF, c, st + 2 + PF);
                                        __builtin_amdgcn_sched_barrier(0);
                                    }
                            }
                }
                pad(st + 2, to);
                __syncthreads();
                if (++st >= stages) goto done;
            }
        }
    done:;
    }

    // Hands every output of the tile to put(row, column, value): row and
    // column within the block's tile.
    template <class F>
    static __device__ __forceinline__ void each(const acc_t (&acc)[TM][TN], int t, F put) {
        const int lane = t & 63, w = t >> 6, wm = w / WN, wn = w % WN;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < M::NR; ++r)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    put(PA::out(wm, i, M::row(r, lane)), PB::out(wn, j, lane % MF), acc[i][j][r]);
    }
};

// ---- tiles -------------------------------------------------------------------------
// Tile shapes and the time of a round of one block per CU on MI355X, operands
// in cache: ns per k-step (the matrix instructions alone need 53 / 13.2 / 3.3)
// and, for its first loads and its outputs' write, us per round:
//   128x128, 32x32x2, KC 32   60, 7.5 (4 blocks per CU, 4096^3: 978-986 us, 140 TFLOP/s)
//   64x64,   32x32x2, KC 32   16.7, 1.3 (2 per CU, 512x4096x4096: 134-137 us)
//   32x32, 16x64, 64x16, 16x16x4, KC 64   6.1 (1 per CU), 5.3 per further round; 0.5
//            (512x4096x16 24.5 us, 16x4096x4096 25 us)
// The one with the least total is taken: large tiles waste what a ragged edge
// or an unfilled round leaves idle, small ones read each operand more often.
// A 128x128 tile writes its 64 KiB at the end, with no second block on its CU
// to multiply meanwhile, so short reductions take 64x64 ones (us, 128x128 ->
// 64x64: 2048x4096 outputs of k = 64 21.4 -> 17.7, 128 28.8 -> 26.0, 256 43.3 ->
// 40.6; at 2048x2048 of k = 512 38.5 against 41.1, so 128x128 stays), and 64x64
// rather than 32x32 (700x3000 of k = 64 9.7 -> 7.6, a gradient of k = 20 11.4 -> 7.3).  Over
// 177 products and gradients of k = 20 .. 2048 the choice is within 0.5 % of
// the best tile on average, 6 % without the time per round, and never more
// than 0.4 % slower than without it.
enum ChainShape { CHAIN_128, CHAIN_64, CHAIN_32, CHAIN_16x64, CHAIN_64x16 };
struct ChainTiles {
    ChainShape shape;
    int64_t rows, cols;  // tiles along m and n
};
inline ChainTiles chain_tiles(int64_t m, int64_t n, int64_t k, int num_cus) {
    struct Cand {
        ChainShape shape;
        int bm, bn;
        double first, more, round;
    };
    static constexpr Cand cands[] = {{CHAIN_128, 128, 128, 60, 60, 7.5},  {CHAIN_64, 64, 64, 16.7, 16.7, 1.3},
                                     {CHAIN_32, 32, 32, 6.1, 5.3, 0.5},   {CHAIN_16x64, 16, 64, 6.2, 5.4, 0.5},
                                     {CHAIN_64x16, 64, 16, 6.2, 5.4, 0.5}};
    ChainTiles best{};
    double cost = 0;
    for (const Cand &c : cands) {
        const int64_t r = cdiv(m, c.bm), q = cdiv(n, c.bn);
        const double rounds = (double)cdiv(r * q, num_cus);
        const double t = (c.first + c.more * (rounds - 1)) * (double)k * 1e-3 + c.round * rounds;
        if (&c == cands || t < cost) {
            best = {c.shape, r, q};
            cost = t;
        }
    }
    return best;
}

// bm * 1000 + bn of a choice (for the tests).
inline int chain_tile_id(const ChainTiles &t) {
    switch (t.shape) {
    case CHAIN_128: return 128128;
    case CHAIN_64: return 64064;
    case CHAIN_32: return 32032;
    case CHAIN_16x64: return 16064;
    case CHAIN_64x16: return 64016;
    }
    return -1;
}

// Tile of block `id` among rows x cols tiles: the blocks an XCD runs (ids
// round-robin over 8) take consecutive tiles, in groups of 8 tile rows walked
// column by column, so that they share operand panels in that XCD's L2.
__device__ __forceinline__ void chain_tile_of(uint32_t id, uint32_t rows, uint32_t cols, uint32_t &tr, uint32_t &tc) {
    const uint32_t total = rows * cols, per = total / 8, rem = total % 8, x = id % 8;
    const uint32_t tile = x * per + min(x, rem) + id / 8;
    const uint32_t grp = tile / (8 * cols), in = tile % (8 * cols), h = min(rows - grp * 8, 8u);
    tr = grp * 8 + in % h;
    tc = in / h;
}

}  // namespace rq
