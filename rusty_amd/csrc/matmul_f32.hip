// f32 matmul family: the reference's per-token GEMMs on an f32 weight.
//
//   MM_AB  <- rusty-backend/src/kernels.wgsl:7-54    (`matmul_tiled`, C = A.B)
//   MM_ABT <- rusty-backend/src/kernels.wgsl:234-242 (`matmul_bt`,    C = A.B^T)
//   MM_ATB <- rusty-backend/src/kernels.wgsl:244-252 (`matmul_at`,    C = A^T.B)
//
// Every output is one f32 accumulator updated in ascending k with a fused
// multiply-add, the order all three WGSL kernels use, so results are
// bit-identical to a sequential k-ascending fma loop regardless of tiling.
// Most calls run on the f32 matrix cores (matmul_mfma.hpp), which keep that
// arithmetic; the VALU kernels below serve what they are faster at (see
// route()): the tiled one products of a few k-steps, the chains a few outputs
// over a long k.
//
// The tiled kernel: 64x64 tiles per 256-thread block with 4x4 outputs per
// thread; operands are staged through LDS k-major so the inner loop reads
// broadcast rows.  Out-of-range rows/columns/k load as zero, which leaves
// every in-range accumulator unchanged.
#include <type_traits>

#include "common.hpp"
#include "lds_dma.hpp"
#include "matmul_mfma.hpp"

namespace rq {
namespace {

constexpr int BM = 64, BN = 64, BK = 16, TH = 256;

// Operand loads without branches or selects on the loaded value: an
// out-of-range element loads element 0 (the callers never load from an empty
// operand) and is replaced by zero only when it is staged, after the loads of
// a whole step are in flight.  A branch around each load made the compiler
// wait for every load at its join (s_waitcnt vmcnt(0) per element), and a
// select right after the load waits for it just the same.
// logical A[r, c] with r < m, c < k; A stored [k, m] for MM_ATB
template <int V>
__device__ __forceinline__ bool in_a(int64_t r, int64_t c, int64_t m, int64_t k) { return r < m && c < k; }
template <int V>
__device__ __forceinline__ float raw_a(const float *a, int64_t r, int64_t c, int64_t m, int64_t k) {
    return a[in_a<V>(r, c, m, k) ? (V == MM_ATB ? c * m + r : r * k + c) : 0];
}
// logical B[r, c] with r < k, c < n; B stored [n, k] for MM_ABT
template <int V>
__device__ __forceinline__ bool in_b(int64_t r, int64_t c, int64_t k, int64_t n) { return r < k && c < n; }
template <int V>
__device__ __forceinline__ float raw_b(const float *b, int64_t r, int64_t c, int64_t k, int64_t n) {
    return b[in_b<V>(r, c, k, n) ? (V == MM_ABT ? c * k + r : r * n + c) : 0];
}

template <int V>
__global__ __launch_bounds__(TH) void k_matmul_f32(const float *__restrict__ a, const float *__restrict__ b,
                                                   float *__restrict__ out, int64_t m, int64_t k, int64_t n) {
    __shared__ float As[BK][BM + 1];
    __shared__ float Bs[BK][BN + 1];
    const int t = threadIdx.x;
    const int tx = t % 16, ty = t / 16;
    const int64_t m0 = (int64_t)blockIdx.y * BM, n0 = (int64_t)blockIdx.x * BN;

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;

    // A tile BM x BK and B tile BK x BN, each thread's 4 + 4 elements coalesced
    // along the operand's contiguous dimension; the next step's elements are
    // loaded into registers before the current step's fmas run (all of them
    // in flight at once: stored to LDS one by one as they arrived, each load
    // had waited for the previous one).
    float ra[4], rb[4];
    auto a_at = [&](int i, int &r, int &c) {
        if constexpr (V == MM_ATB) { r = t % 64; c = t / 64 + 4 * i; }
        else { c = t % 16; r = t / 16 + 16 * i; }
    };
    auto b_at = [&](int i, int &r, int &c) {  // r: k within the step, c: column
        if constexpr (V == MM_ABT) { r = t % 16; c = t / 16 + 16 * i; }
        else { c = t % 64; r = t / 64 + 4 * i; }
    };
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int r, c;
            a_at(i, r, c);
            ra[i] = raw_a<V>(a, m0 + r, k0 + c, m, k);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int r, c;
            b_at(i, r, c);
            rb[i] = raw_b<V>(b, k0 + r, n0 + c, k, n);
        }
    };
    if (k > 0) load(0);
    for (int64_t k0 = 0; k0 < k; k0 += BK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int r, c;
            a_at(i, r, c);
            As[c][r] = in_a<V>(m0 + r, k0 + c, m, k) ? ra[i] : 0.0f;
            b_at(i, r, c);
            Bs[r][c] = in_b<V>(k0 + r, n0 + c, k, n) ? rb[i] : 0.0f;
        }
        __syncthreads();
        if (k0 + BK < k) load(k0 + BK);
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
            const int64_t r = m0 + ty + 16 * i, c = n0 + tx + 16 * j;
            if (r < m && c < n) out[r * n + c] = acc[i][j];
        }
}

// One 16x16 tile of outputs over a long k (a LoRA adapter's x . A at decode)
// is a single chain of dependent fmas whatever runs it: a
// block owns a TR x TC output tile, one output per thread (TR * TC = 256),
// and the k-ascending fma chain per output runs over k-chunks of KC
// staged in LDS by all the block's threads (coalesced along the operand's
// contiguous dimension); the next chunk's loads are in registers before the
// current chunk's chains run.  A is staged [TR][KC + 4] and B transposed,
// [TC][KC + 4] (16-byte rows: four k-steps of each operand per LDS read).
//
// The chunk loads are buffer loads at one per-thread 32-bit offset per
// operand plus a per-element stride held in scalar registers, with no bounds
// test: a position past the operand reads as zero (the buffer's size), and
// one past a row's end lands on a value of a row or column whose output is
// never stored, or on k past K, which no chain reads (a partial chunk's
// chains stop at K).  Per-element 64-bit addresses with clamped indices kept
// some 130 VGPRs live across the chunk loop, and the compiler moved the
// arriving values into AGPRs before the chains -- a wait for the loads it
// had just issued, so every chunk paid a memory round trip (1 x 4096 x 16:
// 45 us).  The host keeps every offset below 2^32 (chain_fits).  Waves whose
// rows all lie past m skip the chains (m = 1 with 16 rows per block: 3 of 4).
__device__ __forceinline__ float bload(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

template <int TC>
constexpr int chain_kc() { return TC == 16 ? 512 : 256; }  // 40-64 KiB of LDS per chunk

// AH: A holds fp16 values (MM_AB only), loaded as 2-byte elements and
// widened exactly when staged -- the f32 matmul of the widened copy, without
// the copy (a LoRA adapter's x . A on fp16 activations).
template <int V, int TC, bool AH = false>
__global__ __launch_bounds__(TH) void k_matmul_f32_chain(const void *__restrict__ a, const float *__restrict__ b,
                                                         float *__restrict__ out, int64_t m, int64_t k, int64_t n) {
    static_assert(!AH || V == MM_AB, "fp16 A: C = A.B only");
    constexpr uint32_t EA = AH ? 2u : 4u;  // bytes per A element
    constexpr int TR = TH / TC;
    constexpr int KC = chain_kc<TC>();
    constexpr int P = KC / TH;                       // chunk rows of TH elements per contiguous row piece
    constexpr int AS = KC + 4;                       // padded A row (floats)
    constexpr int NA = TR * KC / TH, NB = KC * TC / TH;  // chunk elements per thread
    constexpr int G = 32;                            // k-steps per register set of the chains
    // (+ G: the chains' reads one register set past the chunk stay inside the arrays)
    __shared__ __attribute__((aligned(16))) float As[TR * AS + G];
    __shared__ __attribute__((aligned(16))) float Bs[TC * AS + G];
    const int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int64_t r0 = (int64_t)blockIdx.y * TR, c0 = (int64_t)blockIdx.x * TC;
    const int tr = t / TC, tc = t % TC;  // this thread's output
    const uint32_t K = (uint32_t)k, M = (uint32_t)m, N = (uint32_t)n;
    const auto ra_ = make_rsrc(a, (uint32_t)(m * k * EA)), rb_ = make_rsrc(b, (uint32_t)(k * n * 4));
    // Element e of this thread in a chunk: LDS index and byte offset from the
    // thread's base offset (uniform per e); the bases advance by a chunk.
    //  A [m, k] (A [k, m] for MM_ATB), B [k, n] (B [n, k] for MM_ABT).
    uint32_t va, vb, da, db;
    if constexpr (V == MM_ATB) {
        va = ((uint32_t)(t / TR) * M + (uint32_t)r0 + (uint32_t)(t % TR)) * 4u;
        da = (uint32_t)KC * M * 4u;
    } else {
        va = ((uint32_t)r0 * K + (uint32_t)t) * EA;
        da = (uint32_t)KC * EA;
    }
    if constexpr (V == MM_ABT) {
        vb = ((uint32_t)c0 * K + (uint32_t)t) * 4u;
        db = (uint32_t)KC * 4u;
    } else {
        vb = ((uint32_t)(t / TC) * N + (uint32_t)c0 + (uint32_t)(t % TC)) * 4u;
        db = (uint32_t)KC * N * 4u;
    }
    auto a_soff = [&](int e) -> uint32_t {
        if constexpr (V == MM_ATB) return (uint32_t)(TC * e) * M * 4u;
        else return (uint32_t)(e / P) * K * EA + (uint32_t)(e % P) * (TH * EA);
    };
    auto a_lds = [&](int e) {
        if constexpr (V == MM_ATB) return (t % TR) * AS + t / TR + TC * e;
        else return (e / P) * AS + t + TH * (e % P);
    };
    auto b_soff = [&](int e) -> uint32_t {
        if constexpr (V == MM_ABT) return (uint32_t)(e / P) * K * 4u + (uint32_t)(e % P) * (TH * 4u);
        else return (uint32_t)(TR * e) * N * 4u;
    };
    auto b_lds = [&](int e) {
        if constexpr (V == MM_ABT) return (e / P) * AS + t + TH * (e % P);
        else return (t % TC) * AS + t / TC + TR * e;
    };
    float ra[NA], rb[NB];  // AH: ra holds the raw fp16 bits
    auto load = [&]() {
#pragma unroll
        for (int e = 0; e < NA; ++e) {
            if constexpr (AH)
                ra[e] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(ra_, va, a_soff(e), 0));
            else
                ra[e] = bload(ra_, va, a_soff(e));
        }
#pragma unroll
        for (int e = 0; e < NB; ++e) rb[e] = bload(rb_, vb, b_soff(e));
        va += da;
        vb += db;
    };
    auto stage = [&]() {
#pragma unroll
        for (int e = 0; e < NA; ++e) {
            if constexpr (AH)
                As[a_lds(e)] = (float)__builtin_bit_cast(_Float16, (uint16_t)__builtin_bit_cast(uint32_t, ra[e]));
            else
                As[a_lds(e)] = ra[e];
        }
#pragma unroll
        for (int e = 0; e < NB; ++e) Bs[b_lds(e)] = rb[e];
    };
    // this wave's rows: (64 / TC) from 64 wave / TC
    const bool idle = r0 + 64 * wave / TC >= m;
    float acc = 0.0f;
    if (k > 0) load();
    for (int64_t k0 = 0; k0 < k; k0 += KC) {
        stage();
        __syncthreads();
        if (k0 + KC < k) load();  // in flight while this chunk's chains run
        const float *ar = As + tr * AS, *bc = Bs + tc * AS;
        if (idle) {
        } else if (k0 + KC <= k) {
            // two named register sets of G k-steps: the next set's LDS reads are
            // issued (unconditionally) before the current set's fmas (a
            // scheduling barrier keeps the compiler from sinking them below)
            float xa0[G], xb0[G], xa1[G], xb1[G];
            auto rd = [&](float *xa, float *xb, int kk) {
#pragma unroll
                for (int i = 0; i < G; i += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(ar + kk + i);
                    const float4 u = *reinterpret_cast<const float4 *>(bc + kk + i);
                    xa[i] = v.x;
                    xa[i + 1] = v.y;
                    xa[i + 2] = v.z;
                    xa[i + 3] = v.w;
                    xb[i] = u.x;
                    xb[i + 1] = u.y;
                    xb[i + 2] = u.z;
                    xb[i + 3] = u.w;
                }
            };
            auto fm = [&](const float *xa, const float *xb) {
#pragma unroll
                for (int i = 0; i < G; ++i) acc = __builtin_fmaf(xa[i], xb[i], acc);
            };
            rd(xa0, xb0, 0);
            for (int kk = 0; kk < KC; kk += 2 * G) {
                rd(xa1, xb1, kk + G);
                __builtin_amdgcn_sched_barrier(0);
                fm(xa0, xb0);
                rd(xa0, xb0, kk + 2 * G);  // at the chunk's end: read, not used
                __builtin_amdgcn_sched_barrier(0);
                fm(xa1, xb1);
            }
        } else {
            const int kc = (int)(k - k0);
            for (int kk = 0; kk < kc; ++kk) acc = __builtin_fmaf(ar[kk], bc[kk], acc);
        }
        __syncthreads();  // every chain is done with the chunk before it is overwritten
    }
    const int64_t r = r0 + tr, c = c0 + tc;
    if (r < m && c < n) out[r * n + c] = acc;
}

// The same chains for C = A.B^T fed through an LDS ring of NS chunks of KC =
// 256 k-steps filled by global -> LDS DMA (16 bytes per lane, no registers
// held), so NS - 1 chunks are in flight while one is multiplied.  A chain
// advances one dependent fma per 8.4 cycles (MI355X, one wave), 0.9 us per
// chunk, while a chunk's loads take about two: with one chunk in flight (the
// register-staged kernel above) every chunk waited for its data.  Both
// operands keep their rows along k in LDS, as the DMA writes lane pieces
// contiguously: [R][KC + 4], each row's chunk one 1 KiB DMA unit; the chain
// reads four k-steps per ds_read_b128.
// Units of a chunk: TR for A, TC for B, wave w issuing units w, w + 4, ...
// Positions past an operand read as zero or land in rows or k that no stored
// output uses (as above); the dummy DMAs of chunks past K use an offset
// beyond every resource (operands < 2 GiB, chain_fits).  Requires 16-byte
// aligned operands and row pitches (ring_ok).
constexpr int RKC = 256;
constexpr uint32_t kOOBf = 0x80000000u;  // past every operand resource (operands < 2 GiB)
template <int TC>
struct RingShape {
    static constexpr int TR = TH / TC;
    static constexpr int SA = TR * (RKC + 4), SB = TC * (RKC + 4);  // floats per stage
    static constexpr int ST = SA + SB;
    static constexpr int NS = 4 * ST * 4 <= 140 * 1024 ? 4 : 3;
    static constexpr int OPS = (TR + TC) / 4;  // DMA units per wave per chunk
    static_assert(3 * ST * 4 <= 140 * 1024 && (TR + TC) % 4 == 0, "ring does not fit");
};

template <int TC>
__global__ __launch_bounds__(TH) void k_matmul_f32_ring(const float *__restrict__ a, const float *__restrict__ b,
                                                        float *__restrict__ out, int64_t m, int64_t k, int64_t n) {
    using RS = RingShape<TC>;
    constexpr int TR = RS::TR, NS = RS::NS, OPS = RS::OPS, SA = RS::SA, ST = RS::ST, AS = RKC + 4;
    constexpr int G = 32;
    // (+ G: the chains' reads one register set past a chunk stay inside the ring)
    __shared__ __attribute__((aligned(1024))) float ring[NS * ST + G * (TR + TC)];
    const int t = threadIdx.x, lane = t % 64;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int64_t r0 = (int64_t)blockIdx.y * TR, c0 = (int64_t)blockIdx.x * TC;
    const int tr = t / TC, tc = t % TC;
    const uint32_t K = (uint32_t)k;
    const auto rsa = make_rsrc(a, (uint32_t)(m * k * 4)), rsb = make_rsrc(b, (uint32_t)(k * n * 4));
    const uint32_t ring0 = lds_addr(&ring[0]);
    const int nck = (int)((k + RKC - 1) / RKC);

    // Byte offset of this lane's piece of row i of a panel in chunk c: k = c KC + 4 lane.
    auto off_k = [&](uint32_t row0, uint32_t ld, int i, int c) {
        return (((row0 + (uint32_t)i) * ld + (uint32_t)(c * RKC)) + 4u * (uint32_t)lane) * 4u;
    };
    auto issue = [&](int c) {
        const int s = c % NS;
        const bool live = c < nck;
#pragma unroll
        for (int q = 0; q < OPS; ++q) {
            const int u = wave + 4 * q;  // wave-uniform
            if (u < TR) {
                const uint32_t dst = ring0 + (uint32_t)(s * ST) * 4u + (uint32_t)(u * AS) * 4u;
                const uint32_t off = off_k((uint32_t)r0, K, u, c);
                dma16(rsa, dst, live ? off : kOOBf);
            } else {
                const int i = u - TR;
                const uint32_t dst = ring0 + (uint32_t)(s * ST + SA) * 4u + (uint32_t)(i * AS) * 4u;
                const uint32_t off = off_k((uint32_t)c0, K, i, c);
                dma16(rsb, dst, live ? off : kOOBf);
            }
        }
    };

    const bool idle = r0 + 64 * wave / TC >= m;  // every row of this wave lies past m
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < NS - 1; ++c) issue(c);
    for (int c = 0; c < nck; ++c) {
        wait_vmcnt<(NS - 2) * OPS>();  // this wave's units of chunk c have landed
        __syncthreads();               // ... and every wave's; chunk c - 1 is no longer read
        issue(c + NS - 1);             // into chunk c - 1's stage
        if (idle) continue;
        const float *sa = ring + (c % NS) * ST, *sb = sa + SA;
        auto a_at = [&](int kk) -> const float * { return sa + tr * AS + kk; };
        auto b_at = [&](int kk) -> const float * { return sb + tc * AS + kk; };
        const int64_t k0 = (int64_t)c * RKC;
        if (k0 + RKC <= k) {
            float xa0[G], xb0[G], xa1[G], xb1[G];
            auto rd = [&](float *xa, float *xb, int kk) {
#pragma unroll
                for (int i = 0; i < G; i += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(a_at(kk + i));
                    xa[i] = v.x;
                    xa[i + 1] = v.y;
                    xa[i + 2] = v.z;
                    xa[i + 3] = v.w;
                    const float4 u = *reinterpret_cast<const float4 *>(b_at(kk + i));
                    xb[i] = u.x;
                    xb[i + 1] = u.y;
                    xb[i + 2] = u.z;
                    xb[i + 3] = u.w;
                }
            };
            auto fm = [&](const float *xa, const float *xb) {
#pragma unroll
                for (int i = 0; i < G; ++i) acc = __builtin_fmaf(xa[i], xb[i], acc);
            };
            rd(xa0, xb0, 0);
            for (int kk = 0; kk < RKC; kk += 2 * G) {
                rd(xa1, xb1, kk + G);
                __builtin_amdgcn_sched_barrier(0);
                fm(xa0, xb0);
                rd(xa0, xb0, kk + 2 * G);  // at the chunk's end: read, not used
                __builtin_amdgcn_sched_barrier(0);
                fm(xa1, xb1);
            }
        } else {
            const int kc = (int)(k - k0);
            for (int kk = 0; kk < kc; ++kk) acc = __builtin_fmaf(*a_at(kk), *b_at(kk), acc);
        }
    }
    wait_vmcnt<0>();  // no DMA in flight past this point
    const int64_t r = r0 + tr, c = c0 + tc;
    if (r < m && c < n) out[r * n + c] = acc;
}

// Every byte offset the chain kernels form (including the past-the-row ones
// above, up to a chunk and a tile beyond each operand) stays below 2^31.
bool chain_fits(int64_t m, int64_t k, int64_t n) {
    const int64_t lim = (int64_t)1 << 29;  // floats
    return (m + 64) * (k + 1024) < lim && (k + 1024) * (n + 128) < lim;
}

// The ring kernel's 16-byte DMA pieces: aligned operands, rows a multiple of
// 4 floats long.
bool ring_ok(const float *a, const float *b, int64_t k) { return aligned(a, 16) && aligned(b, 16) && k % 4 == 0; }

int launch_ring(const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, hipStream_t s) {
    const int tc = n > 16 ? 32 : (n > 8 ? 16 : 8);
    const int64_t gx = cdiv(n, tc), gy = cdiv(m, TH / tc);
    if (gx > 0x7fffffff || gy > 65535)
        return fail(RQ_ERR_SHAPE, "matmul grid too large (m=%lld n=%lld)", (long long)m, (long long)n);
    const dim3 grid((unsigned)gx, (unsigned)gy);
    switch (tc) {
    case 32: hipLaunchKernelGGL((k_matmul_f32_ring<32>), grid, dim3(TH), 0, s, a, b, out, m, k, n); break;
    case 16: hipLaunchKernelGGL((k_matmul_f32_ring<16>), grid, dim3(TH), 0, s, a, b, out, m, k, n); break;
    default: hipLaunchKernelGGL((k_matmul_f32_ring<8>), grid, dim3(TH), 0, s, a, b, out, m, k, n); break;
    }
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

template <int V, bool AH = false>
int launch_chain(const void *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, hipStream_t s) {
    const int tc = n > 8 ? 16 : 8;  // n <= 16 (route)
    const int64_t gx = cdiv(n, tc), gy = cdiv(m, TH / tc);
    if (gx > 0x7fffffff || gy > 65535)
        return fail(RQ_ERR_SHAPE, "matmul grid too large (m=%lld n=%lld)", (long long)m, (long long)n);
    const dim3 grid((unsigned)gx, (unsigned)gy);
    if (tc == 16) hipLaunchKernelGGL((k_matmul_f32_chain<V, 16, AH>), grid, dim3(TH), 0, s, a, b, out, m, k, n);
    else hipLaunchKernelGGL((k_matmul_f32_chain<V, 8, AH>), grid, dim3(TH), 0, s, a, b, out, m, k, n);
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

// Offsets within a panel stay below 2^29 elements (ChainSpan): rows of up to
// 4 M elements along k, 8 M along the outputs.
bool mfma_fits(int v, int64_t m, int64_t k, int64_t n, int num_cus) {
    const int64_t lim = (int64_t)1 << 29;
    if (!((v == MM_ATB ? m * 64 < lim : k * 128 < lim) && (v == MM_ABT ? k * 128 < lim : n * 64 < lim))) return false;
    const ChainTiles t = chain_tiles(m, n, k, num_cus);
    return grid_ok(t.rows * t.cols, MTH);
}
// Which kernel serves a product, measured on MI355X (us, VALU kernels ->
// matrix cores, AB / ABT / ATB unless stated):
//  * k <= 16, or k <= 48 with over 2^21 outputs: the tiled VALU kernel.  Such
//    a product is its output's write, and the tiled kernel's small LDS keeps
//    more blocks in flight (4096x16x4096 18.0 / 17.7 / 16.4 -> 33.3 / 34.1 /
//    31.1, 4096x48x4096 33 -> 41; 512x32x4096 6.3 -> 5.8, 4096x64x4096 40.6 -> 39.5);
//  * A . B^T with at most 65536 outputs and 16-byte pieces: the ring chains,
//    which have more k in flight (8x1024x1024 7.3 -> 8.0, 1x4096x4096 19.4 ->
//    24.8, 16x512x4096 5.0 -> 5.4; even at 16x4096x4096 25.4 -> 25.1);
//  * over 256 k for a single 16x16 tile: the register-staged chains
//    (1x4096x16 22.3 / 18.6 / 22.3 -> 24.4 / 24.2 / 42.2);
//  * 9 to 16 columns over whole k-chunks where an operand loads by element (its
//    rows no multiple of 4), up to 128 rows, or 2048 of k <= 1024: the
//    register-staged chains (17x1024x9 8.0 / 8.1 -> 8.8 / 9.5 AB / ATB,
//    17x4096x9 27.0 / 27.3 -> 27.8 / 30.9, A^T.B 101x1024x16 8.4 -> 9.2; with a
//    ragged k, or more rows over a long k, the other way: 100x1022x9 10.3 -> 9.7 / 9.2,
//    A^T.B 1001x4096x16 31.8 -> 29.6);
//  * everything else: the matrix cores (4096^3 2270 / 2185 / 2223 -> 978 /
//    998 / 966, 512x4096x4096 368 / 329 / 360 -> 146 / 146 / 139, 1024^3 74 /
//    66 / 74 -> 21, 300x1000x777 72 / 64 / 72 -> 10.2 / 9.0 / 10.1,
//    537x2773x2853 241 / 224 / 245 -> 93 / 87 / 101, 8x4096x11008 286 / 254 /
//    292 -> 28, 512x4096x16 27.3 / 26.1 / 28.0 -> 24.7 / 24.7 / 27.0).
enum Route { ROUTE_TILED, ROUTE_CHAIN, ROUTE_RING, ROUTE_MFMA };
template <typename TA>
Route route(int v, const TA *a, const float *b, int64_t m, int64_t k, int64_t n, int num_cus) {
    if (k <= 16 || (k <= 48 && m * n > ((int64_t)1 << 21))) return ROUTE_TILED;
    const bool chain = k > 64 && chain_fits(m, k, n);
    if constexpr (std::is_same_v<TA, float>)
        if (chain && v == MM_ABT && m * n <= 65536 && ring_ok(a, b, k)) return ROUTE_RING;
    const bool one_tile = k > 256 && m <= 16 && n <= 16;
    const bool by_element = n > 8 && n <= 16 && k % chain_kc<16>() == 0 && (m <= 128 || (k <= 1024 && m <= 2048)) &&
                            !(vec_a(v, a, m, k) && vec_b(v, b, k, n));
    if (chain && (one_tile || by_element)) return ROUTE_CHAIN;
    return mfma_fits(v, m, k, n, num_cus) ? ROUTE_MFMA : ROUTE_TILED;
}

}  // namespace

int launch_matmul_f32(int variant, const float *a, const float *b, float *out, int64_t m, int64_t k, int64_t n,
                      int num_cus, hipStream_t s) {
    if (m == 0 || n == 0) return RQ_OK;
    const Route r = route(variant, a, b, m, k, n, num_cus);
    if (r == ROUTE_MFMA) {
        switch (variant) {
        case MM_AB: return launch_mfma_ab(a, b, out, m, k, n, num_cus, s);
        case MM_ABT: return launch_mfma_abt(a, b, out, m, k, n, num_cus, s);
        case MM_ATB: return launch_mfma_atb(a, b, out, m, k, n, num_cus, s);
        default: return fail(RQ_ERR_INVALID_ARGUMENT, "unknown matmul variant %d", variant);
        }
    }
    if (r == ROUTE_RING) return launch_ring(a, b, out, m, k, n, s);
    if (r == ROUTE_CHAIN) {
        switch (variant) {
        case MM_AB: return launch_chain<MM_AB>(a, b, out, m, k, n, s);
        case MM_ABT: return launch_chain<MM_ABT>(a, b, out, m, k, n, s);
        case MM_ATB: return launch_chain<MM_ATB>(a, b, out, m, k, n, s);
        default: return fail(RQ_ERR_INVALID_ARGUMENT, "unknown matmul variant %d", variant);
        }
    }
    const int64_t gx = cdiv(n, BN), gy = cdiv(m, BM);
    if (gx > 0x7fffffff || gy > 65535)
        return fail(RQ_ERR_SHAPE, "matmul grid too large (m=%lld n=%lld)", (long long)m, (long long)n);
    const dim3 grid((unsigned)gx, (unsigned)gy), block(TH);
    // k == 0 runs the same kernel: the k loop is empty and zeros are stored.
    switch (variant) {
    case MM_AB: hipLaunchKernelGGL(k_matmul_f32<MM_AB>, grid, block, 0, s, a, b, out, m, k, n); break;
    case MM_ABT: hipLaunchKernelGGL(k_matmul_f32<MM_ABT>, grid, block, 0, s, a, b, out, m, k, n); break;
    case MM_ATB: hipLaunchKernelGGL(k_matmul_f32<MM_ATB>, grid, block, 0, s, a, b, out, m, k, n); break;
    default: return fail(RQ_ERR_INVALID_ARGUMENT, "unknown matmul variant %d", variant);
    }
    RQ_LAUNCH_CHECK();
    return RQ_OK;
}

// C = A.B with A fp16 (exactly widened) where the kernel of the shape loads
// it as it is; RQ_ERR_UNSUPPORTED (nothing launched) otherwise, and the caller
// widens A itself.
int launch_matmul_f32_ah(const _Float16 *a, const float *b, float *out, int64_t m, int64_t k, int64_t n, int num_cus,
                         hipStream_t s) {
    if (m == 0 || n == 0) return RQ_OK;
    switch (route(MM_AB, a, b, m, k, n, num_cus)) {
    case ROUTE_MFMA: return launch_mfma_ab_f16(a, b, out, m, k, n, num_cus, s);
    case ROUTE_CHAIN: return launch_chain<MM_AB, true>(a, b, out, m, k, n, s);
    default: return RQ_ERR_UNSUPPORTED;
    }
}

}  // namespace rq

// For the tests, no part of the C ABI: the kernel that serves a product with
// 16-byte aligned f32 operands.  0 tiled, 1 register-staged chains, 2 ring
// chains, the tile (bm * 1000 + bn) on the matrix cores.  Host arithmetic.
extern "C" int rusty_matmul_kernel(int variant, int64_t m, int64_t k, int64_t n, int num_cus) {
    using namespace rq;
    const float *aligned16 = reinterpret_cast<const float *>(uintptr_t(64));
    const Route r = route(variant, aligned16, aligned16, m, k, n, num_cus);
    return r == ROUTE_MFMA ? chain_tile_id(chain_tiles(m, n, k, num_cus)) : (int)r;
}
