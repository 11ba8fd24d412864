// attention_pieces.hip.h -- attention of a portion of tokens over F32 keys and values on the bfloat16 matrix instructions: every 32-bit value goes in as three bfloat16 pieces.
//
// The form of attention_tile.hip.h multiplies in 32 bits, 256 products a cycle and CU; 1024 tokens of 16 heads (keys 192, values 128) take 102 us, three times what the products
// need there.  A 32-bit value is the sum of three bfloat16 pieces (8 + 8 + 8 bits, and bfloat16 has its exponents: nothing is scaled, so no row, position or column loses by the size of
// another); six products of pieces, all but those below 2^-25 of the value, take 3/8 of the matrix time.  The first pieces' products have accumulators of their own.  Error of a result,
// 200 tokens behind 300, in 1e-7 of its norm: keys of 72 / 128 / 192 entries 2.5 / 2.6 / 2.7, as 32-bit products 3.9 / 4.6 / 5.3; with channels and positions that tower over the
// others 5.2 / 4.6 / 3.9, as 32-bit products 10.8 / 9.1 / 7.8.  (Two halves with powers of two per row and tile took half the matrix time, 61 us where this takes 76; a range
// of 2^15 within a tile cost bits there, 2^39 the results.)
// Two launches: attention_image_kernel leaves the visible keys and values of every key / value head as tiles of 32 positions, pieces, rows swizzled and values transposed as LDS
// holds them, once for the up to 32 workgroups that read a tile; attention_pieces_kernel copies them straight into LDS.
// A workgroup owns 64 rows (a row = a token and one of the heads that share a key / value head): four waves of 16 rows, times two that take the tiles in turn.  Scores are formed
// transposed (keys x rows), so that a lane's eight weights are the operand of the second product as they stand -- the order of a tile's 32 positions in it is
// [4 g + r, 16 + 4 g + r] for lane group g, and the values' image has that order -- and maximum, sum and rescaling are one number a lane.
// Bounds: the three phases of a pair of tiles one after the other -- scores (matrix instructions, and LDS reads of 36 KB a wave), softmax (vector instructions), weighted values --, 3.9 us
// a pair, and 8 us around them.  LDS holds one pair's keys: the next pair's are requested when all have formed their scores, and arrive behind softmax and weighted values.
// Measured (us, both launches; the 32-bit form): latent, 1024 tokens, 16 heads, keys 192, values 128: 76 (102); 975 tokens behind 1024: 133 (225); window, 1024 tokens, 16
// heads on 4, 128 + 128, capped scores, a sink, a gate: 80 (104); 150 tokens 21 and 21 (24 and 25).
#pragma once
#include "attention_tile.hip.h"
#include "gemm_direct.hip.h"

namespace ntk {

struct PieceAttnArgs {
    TileAttnArgs t;
    uint8_t* image;                 // [G][tiles of the image][tile]
    int n_seen;                     // positions that the last row sees
    int kept_tiles, first_tile, n_tiles, last_key;      // slot s of the image: tile s below kept_tiles, then first_tile + s - kept_tiles; keys t.key0 (0 for the kept ones) .. last_key
};
constexpr int kPieceRows = 64;
template <int DK, int DV> struct PieceTile { static constexpr int K = 3 * 32 * DK * 2, V = 3 * 32 * DV * 2, BYTES = K + V; };      // [a piece of K], three times, [a piece of V], three times

// x = the sum of its pieces, nearest first (8 + 8 + 8 bits).  What is not finite, or rounds to an infinity, comes out of the products as a NaN, and its rows are formed again
__device__ __forceinline__ void pieces_of(const float (&x)[8], uintx4_t (&out)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const uint32_t w = pack_bf16(a, b);
            out[q][i] = w;
            a -= __uint_as_float(w << 16);
            b -= __uint_as_float(w & 0xffff0000u);
        }
    }
}

// grid (tiles, G), 256 threads: eight threads on a position's row.  Bound by its bytes.  VEC: rows and their parts on 16 bytes, sizes in fours
template <int DK, int DV, bool VEC>
__global__ __launch_bounds__(256) void attention_image_kernel(const PieceAttnArgs h) {
    const TileAttnArgs& a = h.t;
    using Tile = PieceTile<DK, DV>;
    constexpr int KP = DK / 64, VP = DV / 64;                 // pieces of eight entries a thread
    __shared__ __attribute__((aligned(16))) uint16_t vt[3][DV * 32];
    const int slot = blockIdx.x, g = blockIdx.y, tid = threadIdx.x, key = tid >> 3, c = tid & 7, dk = a.nA + a.nB;
    const int j = (slot < h.kept_tiles ? slot : h.first_tile + slot - h.kept_tiles) * 32 + key;
    const bool have = j >= a.key0 && j <= h.last_key;
    uint8_t* img = h.image + ((long long)g * h.n_tiles + slot) * Tile::BYTES;
    const long long jr = have ? j : a.key0;
    const float* pa = a.kA + (jr - a.key0) * a.ldA + (long long)g * a.hA;
    const float* pb = a.kB + jr * a.ldB - a.nA;
    const float* pv = a.v + (jr - a.key0) * a.ldV + (long long)g * a.hV;
    float kx[KP][8], vx[VP][8];
    // (no branch around a load: entries past the end re-read the last ones and are cleared)
    auto fetch = [&](float (&v)[8], int d0, int n, const float* first, const float* second, int cut) {
        if constexpr (VEC) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int e = min(d0 + 4 * q, n - 4);
                const float4 t = *reinterpret_cast<const float4*>((e < cut ? first : second) + e);
                v[4 * q] = t.x; v[4 * q + 1] = t.y; v[4 * q + 2] = t.z; v[4 * q + 3] = t.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) { const int e = min(d0 + i, n - 1); v[i] = (e < cut ? first : second)[e]; }
        }
    };
    auto settle = [&](float (&v)[8], int d0, int n) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = have && d0 + i < n ? v[i] : 0.0f;
    };
#pragma unroll
    for (int p = 0; p < KP; ++p) fetch(kx[p], 8 * (c + 8 * p), dk, pa, pb, a.nA);
#pragma unroll
    for (int p = 0; p < VP; ++p) fetch(vx[p], 8 * (c + 8 * p), a.nV, pv, pv, a.nV);
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        uintx4_t u[3];
        settle(kx[p], 8 * (c + 8 * p), dk);
        pieces_of(kx[p], u);
        const int at = key * DK * 2 + (((c + 8 * p) & ~7) | ((c ^ key) & 7)) * 16;
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uintx4_t*>(img + q * 32 * DK * 2 + at) = u[q];
    }
    const int grp = (key >> 2) & 3, ent = ((key >> 4) << 2) | (key & 3);
#pragma unroll
    for (int p = 0; p < VP; ++p) {
        uintx4_t u[3];
        settle(vx[p], 8 * (c + 8 * p), a.nV);
        pieces_of(vx[p], u);
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int d = 8 * (c + 8 * p) + i;
                vt[q][d * 32 + ((grp ^ (d >> 1)) & 3) * 8 + ent] = (uint16_t)(u[q][i / 2] >> (16 * (i & 1)));
            }
    }
    __syncthreads();
    const uintx4_t* s = reinterpret_cast<const uintx4_t*>(&vt[0][0]);
    uintx4_t* o = reinterpret_cast<uintx4_t*>(img + Tile::K);
    for (int i = tid; i < Tile::V / 16; i += 256) o[i] = s[i];
}

// exp(x), x <= 0: 2^(x log2 e) with the rounding of the product made good; 0 from -200 on down to -inf, a NaN stays one
__device__ __forceinline__ float exp_negative(float x) {
    x = x < -200.0f ? -200.0f : x;
    const float t = x * 1.44269504f;
    const float rest = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269504f, -t));
    const float r = __builtin_amdgcn_exp2f(t);
    return fmaf(r, rest * 0.693147181f, r);
}
__device__ __forceinline__ void direct_wait_reads() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }   // this wave's LDS reads are done, and so everywhere in the workgroup; requests stay under way
// over the four lanes of a row (lane % 16)
__device__ __forceinline__ float quad_max(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// VEC: query rows, results and gates on 16 bytes, sizes in fours
template <int DK, int DV, bool VEC, bool BIASED>
__global__ __launch_bounds__(512, 2) void attention_pieces_kernel(const PieceAttnArgs h) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    using Tile = PieceTile<DK, DV>;
    const TileAttnArgs& a = h.t;
    constexpr int KSTEP = DK / 32, VT = DV / 16, NK = Tile::K / 4096, NV = Tile::V / 4096;      // requests of 1 KB a wave
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * Tile::K + 2 * Tile::V];             // keys, then values, [tile of a pair]
    static_assert(4 * (VT * 256 + 128) * 4 <= 2 * Tile::K, "the merge fits");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wave & 3, kh = wave >> 2, i16 = lane & 15, g4 = lane >> 4;
    const int R = a.H / a.G, n_rows = a.T * R, nx = (n_rows + kPieceRows - 1) / kPieceRows, dk = a.nA + a.nB;
    const int g = blockIdx.x % a.G, x = nx - 1 - blockIdx.x / a.G;      // the longest ranges first
    const int row0 = x * kPieceRows, last = min(row0 + kPieceRows, n_rows) - 1;
    auto first_seen = [&](int p) { return a.window <= 0 ? 0 : a.chunks ? (p / a.window) * a.window : max(0, p - a.window + 1); };
    const int jlo = first_seen(a.pos0 + row0 / R), jhi = a.pos0 + last / R;
    // the tiles walked: 0 .. mine - 1 (positions that stay visible), then from `from` to the last
    const int mine = (min(a.keep, jlo) + 31) / 32, from = max(mine, jlo / 32), n_walk = mine + jhi / 32 - from + 1;
    auto tile_of = [&](int n) { return n < mine ? n : from + n - mine; };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const uint8_t* images = h.image + (long long)g * h.n_tiles * Tile::BYTES;
    auto image_of = [&](int n) { const int t = tile_of(n); return images + (long long)(t < h.kept_tiles ? t : h.kept_tiles + t - h.first_tile) * Tile::BYTES; };
    uint32_t lin[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lin[i] = (uint32_t)(rw * 1024 + lane * 16 + i * 4096);
    auto request = [&](uint32_t at, const uint8_t* from_, auto n) {      // N KB for this wave of the four of a tile, 4 KB apart
        constexpr int N = decltype(n)::value;
        static_assert(N == 6 || N == 9, "tiles of 24 or 36 KB");
        direct_load4<4096>(at + rw * 1024, from_, lin[0], lin[1], lin[2], lin[3]);
        if constexpr (N == 6) direct_load2<4096>(at + rw * 1024 + 16384, from_ + 16384, lin[0], lin[1]);
        else {
            direct_load4<4096>(at + rw * 1024 + 16384, from_ + 16384, lin[0], lin[1], lin[2], lin[3]);
            direct_load1(at + rw * 1024 + 32768, from_ + 32768, lin[0]);
        }
    };
    auto request_keys = [&](int i) {
        if (2 * i + kh < n_walk) request(lds0 + kh * Tile::K, image_of(2 * i + kh), std::integral_constant<int, NK>{});
    };
    request_keys(0);
    // this wave's rows, and the lane's
    const int wrow = row0 + rw * 16, rho = wrow + i16, row = min(rho, n_rows - 1);
    const int tok = row / R, pos = rho < n_rows ? a.pos0 + tok : -1, head = g * R + row - tok * R, lo = pos >= 0 ? first_seen(pos) : 0;
    const int wave_last = min(wrow + 15, n_rows - 1), wave_hi = wrow < n_rows ? a.pos0 + wave_last / R : -1, wave_first = a.pos0 + min(wrow, n_rows - 1) / R;
    const int wave_lo = first_seen(wave_first), clear_lo = first_seen(max(wave_hi, 0)), clear_hi = wrow + 15 < n_rows ? wave_first : -1;     // tiles inside need no mask
    const float slope = a.slopes ? a.slopes[head] : 0.0f;
    // queries as operands: row i16, entries 32 s + 8 g4 ..
    uintx4_t qp[KSTEP][3];
    {
        const float* q = a.q + (long long)tok * a.ldq + (long long)head * dk;
        float v[KSTEP][8];
#pragma unroll
        for (int s = 0; s < KSTEP; ++s) {
            const int d0 = 32 * s + 8 * g4;
            if constexpr (VEC) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const float4 t = *reinterpret_cast<const float4*>(q + min(d0 + 4 * c, dk - 4));
                    v[s][4 * c] = t.x; v[s][4 * c + 1] = t.y; v[s][4 * c + 2] = t.z; v[s][4 * c + 3] = t.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[s][i] = q[min(d0 + i, dk - 1)];
            }
        }
#pragma unroll
        for (int s = 0; s < KSTEP; ++s) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[s][i] = 32 * s + 8 * g4 + i < dk ? v[s][i] : 0.0f;
            pieces_of(v[s], qp[s]);
        }
    }
    const bool sunk = (a.sink || a.sinks) && kh == 0;         // (one of a row's waves starts from the sink)
    float mx = sunk ? (a.sinks ? a.sinks[head] : 0.0f) : -INFINITY, l = sunk && g4 == 0 ? 1.0f : 0.0f;
    f4 acc[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    const int n_pairs = (n_walk + 1) / 2;
    for (int i = 0; i < n_pairs; ++i) {
        const int n = 2 * i + kh;
        const bool there = n < n_walk, more = n + 2 < n_walk;
        direct_wait<0>();                                     // this pair's keys are there, the previous one's values used up
        if (there) request(lds0 + 2 * Tile::K + kh * Tile::V, image_of(n) + Tile::K, std::integral_constant<int, NV>{});
        const int j0 = tile_of(n) * 32;
        const bool work = there && j0 <= wave_hi && (j0 + 31 >= wave_lo || j0 < a.keep);
        // ---- scores, transposed: 32 keys x 16 rows.  The first pieces' products have accumulators of their own
        f4 big[2], low[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) big[u] = low[0][u] = low[1][u] = f4{0.f, 0.f, 0.f, 0.f};
        if (work) {
            const uint8_t* ks = lds + kh * Tile::K;
#pragma unroll
            for (int s = 0; s < KSTEP; ++s) {
                const int piece = 4 * s + g4, at = i16 * DK * 2 + ((piece & ~7) | ((piece ^ i16) & 7)) * 16;
                uintx4_t k[3][2];
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int u = 0; u < 2; ++u) k[p][u] = *reinterpret_cast<const uintx4_t*>(ks + p * 32 * DK * 2 + u * 16 * DK * 2 + at);
                auto mul = [&](f4 (&to)[2], int kp, int qq) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) to[u] = TileBf16::mma(k[kp][u], qp[s][qq], to[u]);
                };
                mul(low[0], 0, 2);
                mul(low[1], 1, 1);
                mul(big, 0, 0);
                mul(low[0], 2, 0);
                mul(low[1], 0, 1);
                mul(low[0], 1, 0);
            }
        }
        direct_wait_reads();                                  // everybody has used this pair's keys
        request_keys(i + 1);
        uintx4_t pp[3];
        if (work) {
            // ---- online softmax: this lane's row, keys j0 + 16 u + 4 g4 + r
            float sv[8];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) sv[4 * u + r] = attention_score<BIASED>(a, big[u][r] + (low[0][u][r] + low[1][u][r]), head, pos - (j0 + 16 * u + 4 * g4 + r), slope);
            if (!(j0 >= clear_lo && j0 + 31 <= clear_hi)) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int j = j0 + 16 * (e >> 2) + 4 * g4 + (e & 3);
                    if (!(j <= pos && (j >= lo || j < a.keep))) sv[e] = -INFINITY;
                }
            }
            const float mt = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])), fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
            const float mn = fmaxf(mx, quad_max(mt)), base = mn == -INFINITY ? 0.0f : mn;
            if (__any(mn != mx)) {                            // (a maximum that stays leaves the sums as they are)
                const float corr = exp_negative(mx - base);
                l *= corr;
                mx = mn;
#pragma unroll
                for (int t = 0; t < VT; ++t) acc[t] *= corr;
            }
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                w[e] = exp_negative(sv[e] - base);
                l += w[e];
            }
            pieces_of(w, pp);
        }
        if (more) direct_wait<NK>(); else direct_wait<0>();   // the values are there
        if (work) {
            // ---- weighted values, transposed: DV x 16 rows; the smallest products first
            const uint8_t* vs = lds + 2 * Tile::K + kh * Tile::V + i16 * 64 + ((g4 ^ (i16 >> 1)) & 3) * 16;
#pragma unroll
            for (int t0 = 0; t0 < VT; t0 += 4) {
                uintx4_t v[3][4];
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int t = 0; t < 4; ++t) v[p][t] = *reinterpret_cast<const uintx4_t*>(vs + p * DV * 64 + (t0 + t) * 16 * 64);
                auto mul = [&](int vp, int q) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t0 + t] = TileBf16::mma(v[vp][t], pp[q], acc[t0 + t]);
                };
                mul(2, 0);
                mul(0, 2);
                mul(1, 1);
                mul(1, 0);
                mul(0, 1);
                mul(0, 0);
            }
        }
    }
    // ---- the two waves of sixteen rows meet: the second leaves (max, sum, vectors), the first adds them to its own and stores
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    __syncthreads();
    float* st = reinterpret_cast<float*>(lds) + rw * VT * 256 + lane * 4;                       // [wave][vectors], then [wave][max, sum]
    float* sm = reinterpret_cast<float*>(lds) + 4 * VT * 256 + rw * 128 + lane;
    if (kh > 0) {
        sm[0] = mx;
        sm[64] = l;
#pragma unroll
        for (int t = 0; t < VT; ++t) *reinterpret_cast<f4*>(st + t * 256) = acc[t];
    }
    __syncthreads();
    if (kh > 0 || wrow >= n_rows) return;
    const float m1 = sm[0], mm = fmaxf(fmaxf(mx, m1), -3.4028235e38f);   // a part's weight: exp(its maximum - the row's), over the row's sum
    float w0 = exp_negative(mx - mm), w1 = exp_negative(m1 - mm);
    const float sum = fmaf(w1, sm[64], w0 * l), inv = sum > 0.0f ? a.out_scale / sum : 0.0f;
    w0 *= inv;
    w1 *= inv;
    bool wild = false;
    {
        float* o = a.out + (long long)tok * a.ldo + (long long)head * a.nV + 4 * g4;
        const float* gt = a.gate ? a.gate + (long long)tok * a.ldg + (a.head_gate ? head : head * a.nV + 4 * g4) : nullptr;
        f4 gv[VT];
        if (gt && !a.head_gate) {                             // (all requested ahead of the first use)
#pragma unroll
            for (int t = 0; t < VT; ++t)
                if constexpr (VEC) gv[t] = *reinterpret_cast<const f4*>(gt + min(16 * t, a.nV - 4 - 4 * g4));
                else
#pragma unroll
                    for (int r = 0; r < 4; ++r) gv[t][r] = gt[min(16 * t + r, a.nV - 1 - 4 * g4)];
        }
        const float one = gt && a.head_gate ? 1.0f + expf(-gt[0]) : 1.0f;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            const f4 other = *reinterpret_cast<const f4*>(st + t * 256);
            f4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                y[r] = fmaf(other[r], w1, acc[t][r] * w0);
                wild = wild || (pos >= 0 && 16 * t + 4 * g4 + r < a.nV && !(fabsf(y[r]) < INFINITY));
            }
            if (gt) y = y / (a.head_gate ? f4{one, one, one, one} : f4{1.0f + expf(-gv[t][0]), 1.0f + expf(-gv[t][1]), 1.0f + expf(-gv[t][2]), 1.0f + expf(-gv[t][3])});
            if (pos < 0) continue;
            if constexpr (VEC) { if (16 * t + 4 * g4 < a.nV) *reinterpret_cast<f4*>(o + 16 * t) = y; }
            else
#pragma unroll
                for (int r = 0; r < 4; ++r) if (16 * t + 4 * g4 + r < a.nV) o[16 * t + r] = y[r];
        }
    }
    // A weight of zero does not stop an infinity or a NaN: the products carry such a value to every row of the tile, those that must not see it among them, and a score
    // with one comes out as a NaN.  A row with a result that is not finite is formed again, key by key over what it sees, in 32 bits.
    unsigned long long some = __ballot(wild);
    if (!some) return;
    some |= some >> 32;
    some = (some | some >> 16) & 0xFFFF;
    while (some) {
        const int rr = __builtin_amdgcn_readfirstlane(wrow + __ffsll(some) - 1);
        some &= some - 1;
        const int tt = rr / R, p0 = a.pos0 + tt, l0 = first_seen(p0), hd = g * R + rr % R;
        const float* q = a.q + (long long)tt * a.ldq + (long long)hd * dk;
        const float sl = a.slopes ? a.slopes[hd] : 0.0f;
        float m = a.sinks ? a.sinks[hd] : a.sink ? 0.0f : -INFINITY, total = a.sink || a.sinks ? 1.0f : 0.0f, y[(DV + 63) / 64];
#pragma unroll
        for (int t = 0; t < (DV + 63) / 64; ++t) y[t] = 0.0f;
#pragma unroll 1
        for (int j = l0 > 0 && a.keep <= 0 ? l0 : 0; j <= p0; ++j) {
            if (j < l0 && j >= a.keep) { j = l0 - 1; continue; }
            const float* pa = a.kA + (long long)(j - a.key0) * a.ldA + (long long)g * a.hA;
            const float* pb = a.kB + (long long)j * a.ldB - a.nA;
            const float* pv = a.v + (long long)(j - a.key0) * a.ldV + (long long)g * a.hV;
            float s = 0.0f;
            for (int d = lane; d < dk; d += 64) s = fmaf(q[d], (d < a.nA ? pa : pb)[d], s);
            s = attention_score<BIASED>(a, wave_sum(s), hd, p0 - j, sl);
            const float mn = fmaxf(m, s), corr = m == -INFINITY ? 0.0f : expf(m - mn), p = expf(s - (mn == -INFINITY ? 0.0f : mn));
            m = mn;
            total = fmaf(total, corr, p);
#pragma unroll
            for (int t = 0; t < (DV + 63) / 64; ++t)
                if (64 * t + lane < a.nV) y[t] = fmaf(p, pv[64 * t + lane], y[t] * corr);
        }
        const float iv = total > 0.0f ? a.out_scale / total : 0.0f;
        float* o = a.out + (long long)tt * a.ldo + (long long)hd * a.nV;
        const float* gt = a.gate ? a.gate + (long long)tt * a.ldg + (a.head_gate ? hd : hd * a.nV) : nullptr;
#pragma unroll
        for (int t = 0; t < (DV + 63) / 64; ++t) {
            const int d = 64 * t + lane;
            if (d < a.nV) o[d] = y[t] * iv / (gt ? 1.0f + expf(-gt[a.head_gate ? 0 : d]) : 1.0f);
        }
    }
}

// the tiles that a portion's rows see
static void piece_attention_tiles(const TileAttnArgs& a, PieceAttnArgs& h) {
    const int lo = a.window <= 0 ? 0 : a.chunks ? (a.pos0 / a.window) * a.window : std::max(0, a.pos0 - a.window + 1);
    // (a later row's range starts later: positions that stay visible lie ahead of the LAST row's range)
    const int end = a.pos0 + a.T - 1, hi_lo = a.window <= 0 ? 0 : a.chunks ? (end / a.window) * a.window : std::max(0, end - a.window + 1);
    h.kept_tiles = (std::min(a.keep, hi_lo) + 31) / 32;
    h.first_tile = std::max(h.kept_tiles, lo / 32);
    h.n_tiles = h.kept_tiles + end / 32 - h.first_tile + 1;
    h.last_key = end;
    h.n_seen = end - hi_lo + 1 + std::min(a.keep, hi_lo);
}
static size_t piece_attention_bytes(int tiles, int G, int dk, int dv) {
    if (dk <= 64 || dk > 192 || dv > 128) return 0;
    return (size_t)G * tiles * (dk <= 128 ? PieceTile<128, 128>::BYTES : PieceTile<192, 128>::BYTES);
}
// false: not a portion for this form, or no room; nothing was launched
static bool launch_attention_pieces(const TileAttnArgs& a, void* image, size_t bytes, hipStream_t s) {
    const int dk = a.nA + a.nB;
    PieceAttnArgs h{};
    h.t = a;
    piece_attention_tiles(a, h);
    // Heads that share no keys and values: few tokens behind little context do not earn the image's launch, nor a few tokens of very many heads its bytes, which one or two workgroups
    // read.  us, here and as 32-bit products, keys 192, values 128: 16 heads, 40 tokens 15.5 and 13.9, 100 19.9 and 19.1, 128 20.4 and 21.7, 40 behind 100 22.3 and 24.3; 64 heads, 128
    // behind 100 35 and 33, 32 behind 1000 92 and 99; 128 heads, 64 behind 1000 152 and 102; 96 heads, 160 behind 1000 188 and 166.  Over 504 sizes (1 .. 128 heads, 32 .. 250 tokens behind
    // up to 1000) the choice is behind the other form by 5 % at most.  Two or more heads a key: ahead from 64 rows on at every length, 0.74 .. 0.91 of the time.
    if (a.H == a.G && h.n_seen < 64 + 4 * a.G) return false;
    if (a.H == a.G && a.G > 64 && (long long)a.T * a.G < 20000) return false;
    const size_t need = piece_attention_bytes(h.n_tiles, a.G, dk, a.nV);
    if (!need || !image || ((uintptr_t)image & 15) || bytes < need || a.G > 65535) return false;
    h.image = (uint8_t*)image;
    const bool biased = a.rel || a.slopes || a.softcap > 0.0f;
    const uintptr_t bits = (uintptr_t)a.kA | (uintptr_t)a.v | (a.nB ? (uintptr_t)a.kB : 0) | (uintptr_t)a.q | (uintptr_t)a.out | (a.gate && !a.head_gate ? (uintptr_t)a.gate : 0);
    const bool vec = !((a.nA | a.nB | a.nV | a.hA | a.hV | (int)a.ldA | (int)a.ldB | (int)a.ldV | a.ldq | a.ldo | (a.gate && !a.head_gate ? a.ldg : 0)) & 3) && !(bits & 15);
    const dim3 tiles(h.n_tiles, a.G), grid((a.T * (a.H / a.G) + kPieceRows - 1) / kPieceRows * a.G);
#define NTK_ATTENTION_PIECES(DK, VEC)                                                                                             \
    do {                                                                                                                          \
        hipLaunchKernelGGL((attention_image_kernel<DK, 128, VEC>), tiles, dim3(256), 0, s, h);                                    \
        if (biased) hipLaunchKernelGGL((attention_pieces_kernel<DK, 128, VEC, true>), grid, dim3(512), 0, s, h);                    \
        else hipLaunchKernelGGL((attention_pieces_kernel<DK, 128, VEC, false>), grid, dim3(512), 0, s, h);                          \
    } while (0)
    if (dk <= 128 && vec) NTK_ATTENTION_PIECES(128, true);
    else if (dk <= 128) NTK_ATTENTION_PIECES(128, false);
    else if (vec) NTK_ATTENTION_PIECES(192, true);
    else NTK_ATTENTION_PIECES(192, false);
#undef NTK_ATTENTION_PIECES
    return true;
}

}  // namespace ntk
