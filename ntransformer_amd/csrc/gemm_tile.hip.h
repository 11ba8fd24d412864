// gemm_tile.hip.h -- one tiled product Y[r][n] = sum_k X[r][k] W[n][k] for four precisions of the same walk (F32 activations, dense row-major weights).
//
// A workgroup of WM x WN waves owns a TM x TN tile.  K goes by in chunks of 64 * SUB bytes per weight row: operands travel HBM / L2 -> registers (two chunks
// requested ahead) -> LDS (two buffers, one barrier per chunk) -> matrix cores; activations are converted on their way into LDS.  What bounds such a product at a
// model's sizes (1000 rows, 2000 .. 8000 outputs) is not the matrix pipe but the time a chunk takes to arrive: with one chunk of 32 in flight (the form before this one)
// a 1024 x 2048 x 7488 bf16 product spent 0.85 us per chunk, 240 TF/s.  Hence the two chunks in registers beside the one being multiplied, and the split of K over
// workgroups (`splits`, partial sums to scratch, summed in order by a second launch) where the tiles alone leave CUs idle.
// Measured (us; the form before: 64 x 128 / 128 x 128 tiles, bf16; 64 x 64 vector FMAs, F32): bf16 1024 x 2048 x 7488 200 -> 58 + 7 (540 TF/s), 1024 x 14976 x 2048
// 173 -> 122, 1024 x 2048 x 2048 55 -> 26, 40 x 2048 x 7488 102 -> 14; F32 150 x 2048 x 7488 396 -> 60 (77 TF/s), 150 x 14976 x 2048 337 -> 113.
// The barrier waits for LDS only: a __syncthreads() would also drain the requests that are meant to stay in flight.
#pragma once
#include <type_traits>
#include "common.hip.h"

namespace ntk {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8_t __attribute__((ext_vector_type(8)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {   // round to nearest even (the hardware conversion)
    const bf16x2_t v = __builtin_convertvector(floatx2_t{a, b}, bf16x2_t);
    uint32_t u;
    __builtin_memcpy(&u, &v, 4);
    return u;
}
template <typename T> __device__ __forceinline__ T bits_as(const uintx4_t u) {
    T t;
    static_assert(sizeof(T) == 16, "sixteen bytes");
    __builtin_memcpy(&t, &u, 16);
    return t;
}

struct TileArgs {
    float* Y; int ldy;
    const float* X; int ldx;
    const void* W; long long wstride;               // one matrix per group, wstride elements apart
    const int* offsets; int G;                      // rows [offsets[g], offsets[g + 1]) belong to group g; NULL: one group of T rows
    const int* rows; int row_div;                   // row r reads activation row rows[r] / row_div
    int T, N, K, accumulate, act;
    int splits, k_per_split;                        // K in `splits` pieces of k_per_split (a multiple of the chunk); > 1: sums go to part[split][T][N]
    float* part;
    const float* row_max;                           // TileHalf2: largest |x| of every activation row (no gathered rows then)
};

// ---- the four precisions: WT the stored weight, KE weights per 64 bytes, PIECES how many values stand for one activation.  RUN: the accumulators are added
// onto a second set and start again from zero every RUN inputs (0: one chain, inputs rounded to eight bits dwarf it).  Products with an activation's pieces behind the first go to
// a set of their own, which stays small beside the first's, so that they cost it no roundings.  Error of a product of 3072 / 4096 / 14336 halves against 64 bits, in 1e-7 of the result, for normal
// activations | with channels of 300 times the others: one set, runs of 128 1.52 1.61 2.28 | 1.63 1.75 2.51; so 1.30 1.40 2.14 | 1.43 1.55 2.35; one-token products (sums over 64 lanes)
// 1.42 1.59 2.78 | 1.42 1.59 2.76.  Three bfloat16 pieces of 512 / 2048 / 4096: one set, runs of 256 1.78 1.84 1.91 | 1.86 1.88 1.99; so 0.76 1.00 1.24 | 0.95 1.17 1.40;
// one-token products 0.86 1.22 1.59 | 0.85 1.22 1.59.
struct TileBf16 {                                   // activations rounded to bfloat16
    using WT = uint16_t;
    static constexpr int KE = 32, EP = 8, PIECES = 1, RUN = 0, STEPS = 1;
    static constexpr bool SCALED = false;
    __device__ static void convert(const float (&v)[EP], float, uintx4_t (&out)[PIECES]) {
        out[0] = uintx4_t{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
    }
    __device__ static floatx4_t mma(uintx4_t a, uintx4_t b, floatx4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(bits_as<bf16x8_t>(a), bits_as<bf16x8_t>(b), c, 0, 0, 0); }
    __device__ static floatx4_t step(uintx4_t a, uintx4_t b, floatx4_t c, int) { return mma(a, b, c); }
};
struct TileBf16x3 {                                 // bfloat16 weights, a 32-bit activation as the three bfloat16 values that add up to it
    using WT = uint16_t;
    static constexpr int KE = 32, EP = 8, PIECES = 3, RUN = 128;
    static constexpr bool SCALED = false;
    __device__ static void convert(const float (&v)[EP], float, uintx4_t (&out)[PIECES]) {
        uint32_t u[EP];
#pragma unroll
        for (int i = 0; i < EP; ++i) u[i] = __float_as_uint(v[i]);
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {                  // cut, not rounded: eight bits a piece, nothing overflows; an infinity stays one, a NaN a NaN
#pragma unroll
            for (int i = 0; i < EP / 2; ++i) out[q][i] = (u[2 * i] >> 16) | (u[2 * i + 1] & 0xffff0000u);
#pragma unroll
            for (int i = 0; i < EP; ++i) {
                const float x = __uint_as_float(u[i]), a = __uint_as_float(u[i] & 0xffff0000u);
                u[i] = x == a ? 0u : __float_as_uint(x - a);
            }
        }
    }
    __device__ static floatx4_t mma(uintx4_t a, uintx4_t b, floatx4_t c) { return TileBf16::mma(a, b, c); }
};
struct TileF32 {                                    // everything in 32 bits: v_mfma_f32_16x16x4_f32, component c of both operands' 16 bytes at a time
    using WT = float;
    static constexpr int KE = 16, EP = 4, PIECES = 1, RUN = 256;
    static constexpr bool SCALED = false;
    __device__ static void convert(const float (&v)[EP], float, uintx4_t (&out)[PIECES]) {
        out[0] = uintx4_t{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    }
    static constexpr int STEPS = 4;                     // (matrix instructions of an operand pair)
    __device__ static floatx4_t mma(uintx4_t a, uintx4_t b, floatx4_t c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) c = step(a, b, c, i);
        return c;
    }
    __device__ static floatx4_t step(uintx4_t a, uintx4_t b, floatx4_t c, int i) { return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i]), __uint_as_float(b[i]), c, 0, 0, 0); }
};
// the power of two that brings a row's largest |x| into [2^14, 2^15) (at most 2^125; below 2^15 whatever finite values stand beside an infinity), and its inverse
__device__ __forceinline__ float half_scale(float largest) {
    const int e = (int)(__float_as_uint(largest) >> 23) & 255;
    return __uint_as_float((uint32_t)min(127 + 14 - (e - 127), 252) << 23);
}
__device__ __forceinline__ float half_unscale(float largest) { return __uint_as_float((254u << 23) - __float_as_uint(half_scale(largest))); }
struct TileHalf2 {                                  // IEEE-half weights, a 32-bit activation (times a power of two) as two halves: off by 2^-23 of it, or 2^-39 of its row's largest, at most
    using WT = uint16_t;
    static constexpr int KE = 32, EP = 8, PIECES = 2, RUN = 128, STEPS = 1;
    static constexpr bool SCALED = true;                // rows times half_scale(row_max)
    __device__ static void convert(const float (&v)[EP], float scale, uintx4_t (&out)[PIECES]) {
        halfx8_t hi, lo;
#pragma unroll
        for (int i = 0; i < EP; ++i) {
            const float x = v[i] * scale;
            hi[i] = (_Float16)x;
            const float back = (float)hi[i];
            lo[i] = x == back ? (_Float16)0.0f : (_Float16)(x - back);      // (an infinity stays one)
        }
        __builtin_memcpy(&out[0], &hi, 16);
        __builtin_memcpy(&out[1], &lo, 16);
    }
    __device__ static floatx4_t mma(uintx4_t a, uintx4_t b, floatx4_t c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(bits_as<halfx8_t>(a), bits_as<halfx8_t>(b), c, 0, 0, 0); }
    __device__ static floatx4_t step(uintx4_t a, uintx4_t b, floatx4_t c, int) { return mma(a, b, c); }
};

// group and first row of row tile `t` when every group's rows are cut into tiles of TM (all groups together at most T / TM + G of them); false: past the last tile
__device__ __forceinline__ bool group_tile(const int* offsets, int G, int t, int TM, int& g, int& r0, int& r1) {
    const int lane = threadIdx.x & 63;
    int before = 0;
    for (int base = 0; base < G; base += 64) {
        const int i = base + lane;
        const int a = offsets[min(i, G)], b = offsets[min(i + 1, G)];
        const int mine = i < G ? (b - a + TM - 1) / TM : 0;
        int sum = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) { const int o = __shfl_up(sum, d, 64); if (lane >= d) sum += o; }
        const unsigned long long past = __ballot(before + sum > t);
        if (past) {
            const int l = __ffsll((unsigned long long)past) - 1;
            g = base + l;
            r0 = __builtin_amdgcn_readlane(a, l) + (t - before - __builtin_amdgcn_readlane(sum - mine, l)) * TM;
            r1 = __builtin_amdgcn_readlane(b, l);
            return true;
        }
        before += __builtin_amdgcn_readlane(sum, 63);
    }
    return false;
}

// LDS is visible to the workgroup; requests to global memory stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// grid: (column tiles, row tiles * splits); VEC: every row of X and W starts on 16 bytes and K is a multiple of EP (no piece crosses the end of a row), and the rows of a tile lie within 2^32 entries
// (eight waves and pieces: 128 registers, so that two workgroups share a CU -- weights at 32-bit offsets from the tile's first row and the odd last chunk behind the loop keep them
// there; with twelve of them spilled 200 x 14336 x 4096 halves took 120 us, so 102)
template <class P, int TM, int TN, int SUB, int WM, int WN, bool VEC>
__global__ __launch_bounds__(64 * WM * WN, WM * WN == 8 && P::PIECES > 1 ? 4 : 2) void gemm_tile_kernel(const TileArgs a) {
    using WT = typename P::WT;
    constexpr int BK = P::KE * SUB, EP = P::EP, PIECES = P::PIECES;
    constexpr int THREADS = 64 * WM * WN, PER_ROW = 4 * SUB, RP = THREADS / PER_ROW, PX = TM / RP, PW = TN / RP;      // loader: PER_ROW threads on a row's chunk, RP rows per pass
    constexpr int STRIDE = 64 * SUB + 16;                                                 // bytes of an LDS row: 16 rows of a quarter wave on different banks
    constexpr int MI = TM / (16 * WM), NJ = TN / (16 * WN);
    static_assert(TM % RP == 0 && TN % RP == 0, "whole passes of the loader");
    __shared__ __attribute__((aligned(16))) uint8_t Xs[2][PIECES][TM * STRIDE];
    __shared__ __attribute__((aligned(16))) uint8_t Ws[2][TN * STRIDE];
    const int split = blockIdx.y % a.splits, rt = blockIdx.y / a.splits;
    int g = 0, row_base = rt * TM, r1 = a.T;
    if (a.offsets) { if (!group_tile(a.offsets, a.G, rt, TM, g, row_base, r1)) return; }
    const int n_base = blockIdx.x * TN;
    const int k_begin = split * a.k_per_split, k_end = min(a.K, k_begin + a.k_per_split), n_chunks = (k_end - k_begin + BK - 1) / BK;
    const WT* W = (const WT*)a.W + (long long)g * a.wstride;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave % WM, wn = wave / WM;
    const int lr = tid / PER_ROW, lp = tid % PER_ROW;
    // rows past the end re-read the last one; what they give is not stored
    const float* xrow[PX];
    const WT* wtile = W + (long long)n_base * a.K;
    typename std::conditional<VEC, uint32_t, size_t>::type wrow[PW];
    float scale[PX];
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        const int r = min(row_base + lr + RP * p, r1 - 1), src = a.rows ? a.rows[r] / a.row_div : r;
        xrow[p] = a.X + (long long)src * a.ldx;
        scale[p] = P::SCALED ? half_scale(a.row_max[src]) : 1.0f;
    }
#pragma unroll
    for (int p = 0; p < PW; ++p) wrow[p] = (decltype(wrow[p] + 0))min(lr + RP * p, a.N - 1 - n_base) * a.K;
    struct Chunk { float x[PX][EP]; uintx4_t w[PW]; };
    auto fetch = [&](Chunk& c, int i) {
        const int k = k_begin + i * BK + lp * EP;
        if constexpr (VEC) {
            const int kc = min(k, a.K - EP);            // (a piece behind the end is cleared on its way into LDS)
#pragma unroll
            for (int p = 0; p < PX; ++p)
#pragma unroll
                for (int q = 0; q < EP / 4; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(xrow[p] + kc + 4 * q);
                    c.x[p][4 * q] = v.x; c.x[p][4 * q + 1] = v.y; c.x[p][4 * q + 2] = v.z; c.x[p][4 * q + 3] = v.w;
                }
#pragma unroll
            for (int p = 0; p < PW; ++p) c.w[p] = *reinterpret_cast<const uintx4_t*>(wtile + (wrow[p] + (uint32_t)kc));
        } else {
#pragma unroll
            for (int p = 0; p < PX; ++p)
#pragma unroll
                for (int j = 0; j < EP; ++j) c.x[p][j] = k + j < k_end ? xrow[p][k + j] : 0.0f;
#pragma unroll
            for (int p = 0; p < PW; ++p) {
                if constexpr (sizeof(WT) == 2) {
                    uint32_t v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = k + j < k_end ? (uint32_t)wtile[wrow[p] + k + j] : 0u;
                    c.w[p] = uintx4_t{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) c.w[p][j] = k + j < k_end ? __float_as_uint((float)wtile[wrow[p] + k + j]) : 0u;
                }
            }
        }
    };
    auto store = [&](const Chunk& c, int i, int buf) {
        const bool in = !VEC || k_begin + i * BK + lp * EP < k_end;
        const uintx4_t zero{0u, 0u, 0u, 0u};
#pragma unroll
        for (int p = 0; p < PX; ++p) {
            uintx4_t u[PIECES];
            P::convert(c.x[p], scale[p], u);
#pragma unroll
            for (int q = 0; q < PIECES; ++q) *reinterpret_cast<uintx4_t*>(&Xs[buf][q][(lr + RP * p) * STRIDE + lp * 16]) = in ? u[q] : zero;
        }
#pragma unroll
        for (int p = 0; p < PW; ++p) *reinterpret_cast<uintx4_t*>(&Ws[buf][(lr + RP * p) * STRIDE + lp * 16]) = in ? c.w[p] : zero;
    };
    floatx4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    constexpr bool SEP = PIECES > 1;
    floatx4_t low[SEP ? MI : 1][SEP ? NJ : 1];
    if constexpr (SEP)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) low[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    constexpr int RUN_CHUNKS = P::RUN / BK;
    static_assert(RUN_CHUNKS % 2 == 0, "a run ends with a pair of chunks");
    floatx4_t total[RUN_CHUNKS ? MI : 1][RUN_CHUNKS ? NJ : 1];
    if constexpr (RUN_CHUNKS > 0)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) total[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto end_run = [&]() {
        if constexpr (RUN_CHUNKS > 0)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) { total[i][j] += acc[i][j]; acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
    };
    const int frag = (lane & 15) * STRIDE + (lane >> 4) * 16;
    auto multiply = [&](int buf) {
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            uintx4_t wf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) wf[j] = *reinterpret_cast<const uintx4_t*>(&Ws[buf][(wn * (TN / WN) + j * 16) * STRIDE + s * 64 + frag]);
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                uintx4_t xf[MI];
#pragma unroll
                for (int i = 0; i < MI; ++i) xf[i] = *reinterpret_cast<const uintx4_t*>(&Xs[buf][q][(wm * (TM / WM) + i * 16) * STRIDE + s * 64 + frag]);
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        if (SEP && q > 0) low[SEP ? i : 0][SEP ? j : 0] = P::mma(xf[i], wf[j], low[SEP ? i : 0][SEP ? j : 0]);
                        else acc[i][j] = P::mma(xf[i], wf[j], acc[i][j]);
                    }
            }
        }
    };
    Chunk c0, c1;
    fetch(c0, 0);
    if (n_chunks > 1) fetch(c1, 1);
    store(c0, 0, 0);
    lds_barrier();
    for (int i = 0; i + 1 < n_chunks; i += 2) {
        if (i + 2 < n_chunks) fetch(c0, i + 2);
        multiply(0);
        store(c1, i + 1, 1);
        lds_barrier();
        if (i + 3 < n_chunks) fetch(c1, i + 3);
        multiply(1);
        if (i + 2 < n_chunks) store(c0, i + 2, 0);
        lds_barrier();
        if constexpr (RUN_CHUNKS > 0) { if ((i + 2) % RUN_CHUNKS == 0) end_run(); }
    }
    if (n_chunks & 1) multiply(0);
    if constexpr (SEP)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] += low[i][j];
    if constexpr (RUN_CHUNKS > 0) {
        end_run();
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = total[i][j];
    }
    // accumulator lane map: row 4 * (lane / 16) + r, column lane % 16
    const int col = n_base + wn * (TN / WN) + (lane & 15), n_left = a.N - col;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = row_base + wm * (TM / WM) + i * 16 + (lane >> 4) * 4;
        float undo[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (P::SCALED)
#pragma unroll
            for (int r = 0; r < 4; ++r) undo[r] = half_unscale(a.row_max[min(row + r, a.T - 1)]);
        if (a.splits > 1) {
            float* y = a.part + ((long long)split * a.T + row) * a.N + col;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < r1 && j * 16 < n_left) y[(long long)r * a.N + j * 16] = acc[i][j][r] * undo[r];
            continue;
        }
        float* y = a.Y + (long long)row * a.ldy + col;
        float old[NJ][4] = {};
        if (a.accumulate)                                   // (what a sum is added onto is requested for a whole strip of tiles before the first store)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) old[j][r] = row + r < r1 && j * 16 < n_left ? y[(long long)r * a.ldy + j * 16] : 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (row + r < r1 && j * 16 < n_left) {
                    float v = acc[i][j][r] * undo[r];
                    if (a.accumulate) v += old[j][r];
                    else if (a.act == 1) { const float p = fmaxf(v, 0.0f); v = p * p; }          // NTK_ACT_RELU2
                    y[(long long)r * a.ldy + j * 16] = v;
                }
    }
}

// Y[r][n] (+)= act(part[0][r][n] + part[1][r][n] + ...), the splits in order; one thread per four columns where rows allow it, else one per column
template <int V>
__global__ __launch_bounds__(256) void gemm_tile_sum_kernel(const TileArgs a) {
    const int n = (blockIdx.x * 256 + threadIdx.x) * V, r = blockIdx.y;
    if (n >= a.N) return;
    const long long plane = (long long)a.T * a.N;
    const float* p = a.part + (long long)r * a.N + n;
    float* y = a.Y + (long long)r * a.ldy + n;
    float s[V] = {}, old[V] = {};
    if (a.accumulate)
#pragma unroll
        for (int j = 0; j < V; ++j) old[j] = y[j];
    for (int i = 0; i < a.splits; i += 4) {                 // four requests under way
        float v[4][V];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float* q = p + plane * min(i + u, a.splits - 1);
            if constexpr (V == 4) { const float4 t = *reinterpret_cast<const float4*>(q); v[u][0] = t.x; v[u][1] = t.y; v[u][2] = t.z; v[u][3] = t.w; }
            else v[u][0] = *q;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u < a.splits)
#pragma unroll
                for (int j = 0; j < V; ++j) s[j] += v[u][j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        if (a.accumulate) s[j] += old[j];
        else if (a.act == 1) { const float q = fmaxf(s[j], 0.0f); s[j] = q * q; }
    }
    if constexpr (V == 4) *reinterpret_cast<float4*>(y) = float4{s[0], s[1], s[2], s[3]};
    else y[0] = s[0];
}

// ---- which tile, and how many pieces of K: the smallest of `chunks x max(alone, workgroups per CU x busy)` + what summing the pieces costs.
// `alone` is what a chunk takes in a workgroup that has a CU for itself (latency), `busy` what a further workgroup on the CU adds (matrix pipe, LDS), both in us and
// measured on the shapes of model layers: 12 .. 1024 rows, 2048 .. 28672 outputs, 512 .. 14336 inputs.  Over 70 such shapes it is
// 2 % behind the best tile and split on average, by more than a tenth in four, by a fifth at most (40 x 28672 x 4096 bf16: 49 us, 41 with 64 x 128 in two pieces).
struct TileForm { int TM, TN, chunk; float alone, busy; };
struct TilePlan { int form, splits; float us; };
static TilePlan plan_tiles(const TileForm* f, int n_forms, int rows, int groups, int N, int K, long long scratch_floats) {
    static const int counts[] = {1, 2, 3, 4, 6, 8, 12, 16};
    TilePlan best{0, 1, 1e30f};
    for (int i = 0; i < n_forms; ++i) {
        // (rows of several groups: on average half a tile of each is empty)
        const int row_tiles = groups > 1 ? rows / f[i].TM + (groups + 1) / 2 : (rows + f[i].TM - 1) / f[i].TM;
        const long long tiles = (long long)row_tiles * ((N + f[i].TN - 1) / f[i].TN);
        const int chunks = (K + f[i].chunk - 1) / f[i].chunk;
        for (int s : counts) {
            if (s > 1 && ((long long)s * rows * N > scratch_floats || chunks < 4 * s)) break;
            const float per_cu = (float)((tiles * s + 255) / 256);
            float us = (float)((chunks + s - 1) / s) * (f[i].alone > per_cu * f[i].busy ? f[i].alone : per_cu * f[i].busy);
            if (s > 1) us += 4.0f + (float)(s + 1) * rows * N * 4.0f / 4e6f;
            if (us < best.us) best = TilePlan{i, s, us};
        }
    }
    return best;
}

static void launch_tile_sum(const TileArgs& a, hipStream_t s) {
    const bool four = a.N % 4 == 0 && a.ldy % 4 == 0 && !(((uintptr_t)a.Y | (uintptr_t)a.part) & 15);
    if (four) hipLaunchKernelGGL((gemm_tile_sum_kernel<4>), dim3((a.N / 4 + 255) / 256, a.T), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((gemm_tile_sum_kernel<1>), dim3((a.N + 255) / 256, a.T), dim3(256), 0, s, a);
}

template <class P, int TM, int TN, int SUB, int WM, int WN, bool VEC>
static int launch_tiles(TileArgs a, int splits, hipStream_t s, bool sum = true) {      // the pieces of K that a.part holds (sum: added up by a launch of their own)
    constexpr int BK = P::KE * SUB;
    const int chunks = (a.K + BK - 1) / BK, per = (chunks + splits - 1) / splits;
    a.k_per_split = per * BK;
    a.splits = (chunks + per - 1) / per;
    const int row_tiles = a.offsets ? a.T / TM + a.G : (a.T + TM - 1) / TM;
    hipLaunchKernelGGL((gemm_tile_kernel<P, TM, TN, SUB, WM, WN, VEC>), dim3((a.N + TN - 1) / TN, row_tiles * a.splits), dim3(64 * WM * WN), 0, s, a);
    if (a.splits > 1 && sum) launch_tile_sum(a, s);
    return a.splits;
}

}  // namespace ntk
