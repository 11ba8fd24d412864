// attention_tile.hip.h -- attention of a portion of tokens over F32 keys and values on the F32 matrix instructions, for the window and the latent mixers.
//
// A workgroup owns 32 rows (a row = a token and one of the R query heads that share a key / value head) and walks the visible keys in tiles of 32: wave (row half, key half)
// holds the queries of 16 rows as operands in registers, forms 16 x 16 scores with v_mfma_f32_16x16x4_f32, keeps the online softmax of its rows over its half of the
// keys and sums 16 x DV values the same way; the halves meet in LDS at the end.  Every product and sum is in 32 bits (a matrix instruction adds four products where
// the vector form before it added one).  What bounded the vector form (lane = key, one LDS read per two FMAs): LDS, 16 TF/s.  Here a 16-byte operand read feeds four
// instructions of 32 cycles; a third of the time is the matrix pipe, the rest the chain scores -> maximum -> exponentials -> weighted values in front of it (two waves
// per SIMD; four key quarters per workgroup instead of two halves: 113 us against 106).  A workgroup's partner on the same CU (256 further on) walks the mirrored range; key / value
// heads go to XCDs as wholes, so that a head's rows meet in one L2.
// Measured (us, before -> after): latent, 1024 tokens, 16 heads, keys 192, values 128: 354 -> 106; 975 tokens behind 1024: 769 -> 235; window, 1024 tokens, 16 heads on 4,
// 128 + 128, capped scores, a sink: 340 -> 109.
#pragma once
#include "common.hip.h"

namespace ntk {

struct TileAttnArgs {
    float* out; int ldo;                               // [T][H][nV]
    const float* q; int ldq;                           // [T][H][nA + nB]
    const float* kA; long long ldA; int nA, hA;        // first part of a key: kA + (j - key0) * ldA + g * hA
    const float* kB; long long ldB; int nB;            // second part, one for all heads: kB + j * ldB
    const float* v; long long ldV; int nV, hV;         // value: v + (j - key0) * ldV + g * hV
    int key0, H, G, pos0, T, window, chunks, keep;     // chunks: `window` is a chunk size; keep: positions 0 .. keep - 1 stay visible
    float scale, softcap, out_scale;
    int sink; const float* sinks;                      // a further key without a value, of score sinks[head] (0 without)
    const float* slopes;
    const float* rel; const int* bucket_of; int n_dist;
    const float* gate; int ldg, head_gate;
};

__device__ __forceinline__ float row16_max(float v) {  // over the sixteen lanes of a row
    v = fmaxf(v, dpp_or_self<DPP_QUAD_1032, 0xF>(v));
    v = fmaxf(v, dpp_or_self<DPP_QUAD_2301, 0xF>(v));
    v = fmaxf(v, dpp_or_self<DPP_ROW_HALF_MIRROR, 0xF>(v));
    return fmaxf(v, dpp_or_self<DPP_ROW_MIRROR, 0xF>(v));
}

// key / value head and row tile of a workgroup (see above); every (g, x) once
__device__ __forceinline__ void attention_place(int id, int G, int nx, int& g, int& x) {
    int slot, slots;
    if (G % 8 == 0) { slot = id / 8; g = (slot / nx) * 8 + id % 8; x = slot % nx; if ((slot / nx) & 1) x = nx - 1 - x; return; }
    if (8 % G == 0 && nx % (8 / G) == 0) {
        const int parts = 8 / G, xcd = id % 8;
        slot = id / 8; slots = nx / parts; g = xcd % G;
        const int half = (slots + 1) / 2, s = slot < half ? slot : slots - 1 - (slot - half);
        x = s * parts + xcd / G;
        return;
    }
    g = id / nx; x = id % nx;
    if (g >= (G + 1) / 2) x = nx - 1 - x;
}

template <bool BIASED>
__device__ __forceinline__ float attention_score(const TileAttnArgs& a, float s, int head, int distance, float slope) {
    s *= a.scale;
    if constexpr (BIASED) {                                   // (each of these for the launch or not at all)
        if (a.rel) s += a.rel[(long long)a.bucket_of[min(max(distance, 0), a.n_dist - 1)] * a.H + head];
        if (a.slopes) s -= slope * (float)distance;
        if (a.softcap > 0.0f) s = a.softcap * tanhf(s / a.softcap);
    }
    return s;
}

// DK, DV: entries of a key and of a value, rounded up (the rest is zero in the operands); VEC: every key / value row is 16-byte aligned and cut in fours
// BIASED: anything but the scale on the scores (bias by distance, slopes, soft cap)
constexpr int KT = 32;                                    // keys of a tile: sixteen for each of the two waves along them
template <int DK, int DV, bool VEC, bool BIASED>
__global__ __launch_bounds__(256, 2) void attention_tile_kernel(const TileAttnArgs a) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int KS = DK + 4, VS = DV + 4, PS = 20, KSTEP = DK / 16, VT = DV / 16;
    constexpr int KU = DK / 32, VU = DV / 32;                 // loader: eight threads on a key's row, 16 bytes each, so many passes
    constexpr int STATE = (8 + 4 * VT) * 64;                  // what a wave leaves for the merge
    constexpr int TILES = KT * (KS + VS) > 2 * STATE ? KT * (KS + VS) : 2 * STATE;
    __shared__ __attribute__((aligned(16))) float tiles[TILES];
    __shared__ __attribute__((aligned(16))) float Ps[4][16 * PS];
    float* Ks = tiles;
    float* Vs = tiles + KT * KS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rh = wave & 1, kh = wave >> 1, i16 = lane & 15, g4 = lane >> 4;
    const int R = a.H / a.G, n_rows = a.T * R, nx = (n_rows + 31) / 32;
    int g, x;
    attention_place(blockIdx.x, a.G, nx, g, x);
    const int row0 = x * 32, last = min(row0 + 32, n_rows) - 1, dk = a.nA + a.nB;
    auto first_seen = [&](int p) { return a.window <= 0 ? 0 : a.chunks ? (p / a.window) * a.window : max(0, p - a.window + 1); };
    const int jlo = first_seen(a.pos0 + row0 / R), jhi = a.pos0 + last / R;
    // the keys walked: 0 .. kept - 1, then jlo .. jhi; number n of the walk is position n, or n + skip from `kept` on
    const int kept = min(a.keep, jlo), skip = jlo - kept, n_keys = kept + jhi - jlo + 1;
    auto key_pos = [&](int n) { return n + (n >= kept ? skip : 0); };
    // the wave's queries as operands: row i16, entries 16 s + 4 g4 ..
    f4 qf[KSTEP];
    {
        const int rho = row0 + rh * 16 + i16;
        const float* q = a.q + (long long)(min(rho, n_rows - 1) / R) * a.ldq + (long long)(g * R + min(rho, n_rows - 1) % R) * dk;
#pragma unroll
        for (int s = 0; s < KSTEP; ++s)
#pragma unroll
            for (int c = 0; c < 4; ++c) { const int d = 16 * s + 4 * g4 + c; const float v = q[min(d, dk - 1)]; qf[s][c] = d < dk ? v : 0.0f; }
    }
    // rows of this lane's scores and sums: 4 g4 + r
    int rpos[4], rhead[4], rlo[4];
    float mx[4], l[4], slope[4];
    f4 acc[VT];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int rho = row0 + rh * 16 + 4 * g4 + r;
        rpos[r] = rho < n_rows ? a.pos0 + rho / R : -1;
        rhead[r] = g * R + rho % R;
        rlo[r] = rpos[r] >= 0 ? first_seen(rpos[r]) : 0;
        slope[r] = a.slopes ? a.slopes[rhead[r]] : 0.0f;
        const bool sunk = (a.sink || a.sinks) && kh == 0;     // (one of a row's waves starts from the sink)
        mx[r] = sunk ? (a.sinks ? a.sinks[rhead[r]] : 0.0f) : -INFINITY;
        l[r] = sunk && i16 == 0 ? 1.0f : 0.0f;                // a lane sums its own columns; the row's sum is formed at the end
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    f4 kreg[KU], vreg[VU];
    const int lk = tid >> 3, lc = tid & 7;
    const bool full = dk == DK && a.nV == DV;
    // (no branch in here: keys past the last re-read it -- their weight is zero -- and entries past the end re-read the last ones and are cleared on their way into LDS)
    auto fetch = [&](int n0) {
        const int j = key_pos(min(n0 + lk, n_keys - 1));
        const float* pa = a.kA + (long long)(j - a.key0) * a.ldA + (long long)g * a.hA;
        const float* pb = a.kB + (long long)j * a.ldB - a.nA;
        const float* pv = a.v + (long long)(j - a.key0) * a.ldV + (long long)g * a.hV;
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int d = 4 * (lc + 8 * u);
            if constexpr (VEC) {
                const int e = min(d, dk - 4);
                kreg[u] = *reinterpret_cast<const f4*>((e < a.nA ? pa : pb) + e);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) { const int e = min(d + c, dk - 1); kreg[u][c] = (e < a.nA ? pa : pb)[e]; }
            }
        }
#pragma unroll
        for (int u = 0; u < VU; ++u) {
            const int d = 4 * (lc + 8 * u);
            if constexpr (VEC) {
                vreg[u] = *reinterpret_cast<const f4*>(pv + min(d, a.nV - 4));
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) vreg[u][c] = pv[min(d + c, a.nV - 1)];
            }
        }
    };
    fetch(0);
    for (int n0 = 0; n0 < n_keys; n0 += KT) {
        __syncthreads();                                      // the previous tile is used up
        if (!full) {
#pragma unroll
            for (int u = 0; u < KU; ++u)
#pragma unroll
                for (int c = 0; c < 4; ++c) if (4 * (lc + 8 * u) + c >= dk) kreg[u][c] = 0.0f;
#pragma unroll
            for (int u = 0; u < VU; ++u)
#pragma unroll
                for (int c = 0; c < 4; ++c) if (4 * (lc + 8 * u) + c >= a.nV) vreg[u][c] = 0.0f;
        }
#pragma unroll
        for (int u = 0; u < KU; ++u) *reinterpret_cast<f4*>(&Ks[lk * KS + 4 * (lc + 8 * u)]) = kreg[u];
#pragma unroll
        for (int u = 0; u < VU; ++u) *reinterpret_cast<f4*>(&Vs[lk * VS + 4 * (lc + 8 * u)]) = vreg[u];
        __syncthreads();
        if (n0 + KT < n_keys) fetch(n0 + KT);                 // behind this tile's products
        // ---- scores of 16 rows x 16 keys
        f4 s4{0.f, 0.f, 0.f, 0.f};
        const float* kf = &Ks[(kh * 16 + i16) * KS + 4 * g4];
#pragma unroll
        for (int s = 0; s < KSTEP; ++s) {
            const f4 k4 = *reinterpret_cast<const f4*>(kf + 16 * s);
#pragma unroll
            for (int c = 0; c < 4; ++c) s4 = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[s][c], k4[c], s4, 0, 0, 0);
        }
        // ---- online softmax; weights to the wave's own LDS
        const int n = n0 + kh * 16 + i16, j = key_pos(n);
        float sv[4], mn[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sv[r] = s4[r] * a.scale;
        if constexpr (BIASED) {                               // (each of these for the launch or not at all)
            if (a.rel)
#pragma unroll
                for (int r = 0; r < 4; ++r) sv[r] += a.rel[(long long)a.bucket_of[min(max(rpos[r] - j, 0), a.n_dist - 1)] * a.H + rhead[r]];
            if (a.slopes)
#pragma unroll
                for (int r = 0; r < 4; ++r) sv[r] -= slope[r] * (float)(rpos[r] - j);
            if (a.softcap > 0.0f)
#pragma unroll
                for (int r = 0; r < 4; ++r) sv[r] = a.softcap * tanhf(sv[r] / a.softcap);
        }
        bool moved = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (!(n < n_keys && j <= rpos[r] && (j >= rlo[r] || j < a.keep))) sv[r] = -INFINITY;
            mn[r] = fmaxf(mx[r], row16_max(sv[r]));
            moved = moved || mn[r] != mx[r];
        }
        if (__any(moved)) {                                   // (a maximum that stays leaves the sums as they are)
            float corr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                corr[r] = mx[r] == -INFINITY ? 0.0f : expf(mx[r] - mn[r]);
                mx[r] = mn[r];
                l[r] *= corr[r];
            }
#pragma unroll
            for (int t = 0; t < VT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][r] *= corr[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float p = expf(sv[r] - (mn[r] == -INFINITY ? 0.0f : mn[r]));       // (0 for a key that is not seen)
            l[r] += p;
            Ps[wave][(4 * g4 + r) * PS + i16] = p;
        }
        __builtin_amdgcn_wave_barrier();                      // (a wave's LDS operations run in order)
        const f4 p4 = *reinterpret_cast<const f4*>(&Ps[wave][i16 * PS + 4 * g4]);
        // ---- weighted values: component c of the weights belongs to key 4 g4 + c
        const float* vf = &Vs[(kh * 16 + 4 * g4) * VS + i16];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int t = 0; t < VT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p4[c], vf[c * VS + 16 * t], acc[t], 0, 0, 0);
        __builtin_amdgcn_wave_barrier();
    }
    // ---- the two waves of a row half meet: the second leaves (max, sum, vectors), the first adds them to its own and stores
#pragma unroll
    for (int r = 0; r < 4; ++r) l[r] = group_sum<16>(l[r]);
    __syncthreads();
    float* st = tiles + rh * STATE + lane;
    if (kh > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) { st[r * 64] = mx[r]; st[(4 + r) * 64] = l[r]; }
#pragma unroll
        for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) st[(8 + 4 * t + r) * 64] = acc[t][r];
    }
    __syncthreads();
    if (kh > 0) return;
    float w0[4], w1[4];                                       // a part's weight: exp(its maximum - the row's), over the row's sum
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float m1 = st[r * 64], mm = fmaxf(mx[r], m1);
        w0[r] = mx[r] == -INFINITY ? 0.0f : expf(mx[r] - mm);
        w1[r] = m1 == -INFINITY ? 0.0f : expf(m1 - mm);
        const float sum = fmaf(w1[r], st[(4 + r) * 64], w0[r] * l[r]);
        const float inv = sum > 0.0f ? a.out_scale / sum : 0.0f;
        w0[r] *= inv;
        w1[r] *= inv;
    }
    uint32_t wild = 0;                                        // results that are not finite: bit 4 t + r
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (rpos[r] < 0) continue;
        const int t0 = rpos[r] - a.pos0;
        float* o = a.out + (long long)t0 * a.ldo + (long long)rhead[r] * a.nV + i16;
        const float* gt = a.gate ? a.gate + (long long)t0 * a.ldg + (a.head_gate ? rhead[r] : rhead[r] * a.nV + i16) : nullptr;
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            if (16 * t + i16 >= a.nV) continue;
            float y = fmaf(st[(8 + 4 * t + r) * 64], w1[r], acc[t][r] * w0[r]);
            if (!(fabsf(y) < INFINITY)) wild |= 1u << (4 * t + r);
            if (gt) y = y / (1.0f + expf(-gt[a.head_gate ? 0 : 16 * t]));
            o[16 * t] = y;
        }
    }
    // A weight of zero does not stop an infinity or a NaN: the products above carry such a value to every row of the tile, those that must not see it among them.  A result that is not
    // finite is formed again, key by key over what its row sees (sixteen lanes a row); ahead of the products, every tile would pay for the question (5 - 11 % of a launch;
    // here 0 - 1 %, 0.3 - 1 us of the shortest).
    if (!__any(wild != 0)) return;
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
        const int rho = row0 + rh * 16 + 4 * g4 + r;
        if (rho >= n_rows) break;
        const int t0 = rho / R, pos = a.pos0 + t0, lo = first_seen(pos), head = g * R + rho % R;
        const float* q = a.q + (long long)t0 * a.ldq + (long long)head * dk;
        const float slope = a.slopes ? a.slopes[head] : 0.0f;
        float m = a.sinks ? a.sinks[head] : a.sink ? 0.0f : -INFINITY, sum = a.sink || a.sinks ? 1.0f : 0.0f, y[VT];
#pragma unroll
        for (int t = 0; t < VT; ++t) y[t] = 0.0f;
#pragma unroll 1
        for (int n = 0; n < n_keys; ++n) {
            const int j = key_pos(n);
            if (j > pos || (j < lo && j >= a.keep)) continue;         // (the sixteen lanes of a row together)
            const float* pa = a.kA + (long long)(j - a.key0) * a.ldA + (long long)g * a.hA;
            const float* pb = a.kB + (long long)j * a.ldB - a.nA;
            const float* pv = a.v + (long long)(j - a.key0) * a.ldV + (long long)g * a.hV;
            float s = 0.0f;
            for (int d = i16; d < dk; d += 16) s = fmaf(q[d], (d < a.nA ? pa : pb)[d], s);
            s = attention_score<BIASED>(a, group_sum<16>(s), head, pos - j, slope);
            const float mn = fmaxf(m, s), corr = m == -INFINITY ? 0.0f : expf(m - mn), p = expf(s - (mn == -INFINITY ? 0.0f : mn));
            m = mn;
            sum = fmaf(sum, corr, p);
#pragma unroll
            for (int t = 0; t < VT; ++t)
                if (16 * t + i16 < a.nV) y[t] = fmaf(p, pv[16 * t + i16], y[t] * corr);
        }
        const float inv = sum > 0.0f ? a.out_scale / sum : 0.0f;
        float* o = a.out + (long long)t0 * a.ldo + (long long)head * a.nV + i16;
        const float* gt = a.gate ? a.gate + (long long)t0 * a.ldg + (a.head_gate ? head : head * a.nV + i16) : nullptr;
#pragma unroll
        for (int t = 0; t < VT; ++t)
            if ((wild >> (4 * t + r)) & 1) o[16 * t] = y[t] * inv / (gt ? 1.0f + expf(-gt[a.head_gate ? 0 : 16 * t]) : 1.0f);
    }
}

// sizes this form has
static bool attention_tile_takes(int dk, int dv) { return dk <= 192 && dv <= 128; }

static void launch_attention_tile(const TileAttnArgs& a, hipStream_t s) {
    const int dk = a.nA + a.nB;
    const bool vec = a.nA % 4 == 0 && a.nB % 4 == 0 && a.nV % 4 == 0 && a.hA % 4 == 0 && a.hV % 4 == 0 && a.ldA % 4 == 0 && a.ldB % 4 == 0 && a.ldV % 4 == 0 &&
                     !(((uintptr_t)a.kA | (uintptr_t)a.v | (a.nB ? (uintptr_t)a.kB : 0)) & 15);
    const dim3 grid((a.T * (a.H / a.G) + 31) / 32 * a.G);
    const bool biased = a.rel || a.slopes || a.softcap > 0.0f;
#define NTK_ATTENTION_TILE(DK, DV, VEC)                                                                                          \
    do {                                                                                                                          \
        if (biased) hipLaunchKernelGGL((attention_tile_kernel<DK, DV, VEC, true>), grid, dim3(256), 0, s, a);                     \
        else hipLaunchKernelGGL((attention_tile_kernel<DK, DV, VEC, false>), grid, dim3(256), 0, s, a);                           \
    } while (0)
    if (!vec) {
        if (dk <= 64 && a.nV <= 64) NTK_ATTENTION_TILE(64, 64, false);
        else NTK_ATTENTION_TILE(192, 128, false);
    } else if (dk <= 64 && a.nV <= 64) NTK_ATTENTION_TILE(64, 64, true);
    else if (dk <= 128) NTK_ATTENTION_TILE(128, 128, true);
    else NTK_ATTENTION_TILE(192, 128, true);
#undef NTK_ATTENTION_TILE
}

}  // namespace ntk
