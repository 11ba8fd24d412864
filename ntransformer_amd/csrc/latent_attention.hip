// latent_attention.hip -- attention over a cache of one normed latent and one rotated key part per position.
//
// What is cached per position and layer run is [latent c (kv_rank) | rotated key part (rot_dim)], F32.  Two ways to the same sums:
//   * expanded (prompt portions): the caller up-projects the cached latents of the visible range into per-head keys and values (two products over
//     the cache rows) and the kernel runs ordinary multi-head attention on them, reading the shared rotated part from the cache rows;
//   * shared (few query tokens, decoding): the query's unrotated part is folded through the key up-projection first (ntk_latent_fold_query), so every
//     head scores against the cache rows themselves, [c | rotated] . [folded q | rotated q]; the weighted sum is taken over c and the value
//     up-projection is applied once afterwards (ntk_latent_unfold_value).  Nothing per head is ever materialised for the cached positions.
// Expanded: a workgroup owns 16 tokens of one head and walks the visible keys in chunks of 64 -- lane = key for the scores (key slabs of 64 entries in
// LDS), online softmax per row in F32, lane = value column for the weighted sum.  Shared: a workgroup owns 16 (token, head) rows and whole tiles of 32
// cache rows; the tiles go round up to 128 workgroups and a second launch merges their (max, sum, vector) states.
#include "attention_pieces.hip.h"
#include "moe_route.hip.h"
#include "../../include/ntk_layers.h"

namespace ntk {

// ------------------------------------------------------------------------------------------------------------------- cache rows and rotation
// one workgroup per token: latent / rms * w and the rotated key part into the cache row, the rotated part of every query head in place.
// Angles in double (position times frequency, then cos / sin), applied in F32.
__global__ __launch_bounds__(256) void latent_prepare_kernel(float* cache, int row, const float* kv, int ldkv, const float* norm_w, float eps, int R, int dr,
                                                             float* q, int ldq, int H, int qd, const double* freq, float mag, int dims, int pos0, int halves) {
    __shared__ float red[16];
    extern __shared__ float cs[];   // [dims / 2] cos, [dims / 2] sin
    const int t = blockIdx.x, pos = pos0 + t;
    const float* src = kv + (long long)t * ldkv;
    float* dst = cache + (long long)pos * row;
    const int half = dims / 2;   // dims <= dr: what lies behind the rotated entries passes unchanged
    for (int i = threadIdx.x; i < half; i += 256) {
        const double a = (double)pos * freq[i];
        cs[i] = (float)(cos(a) * (double)mag);
        cs[half + i] = (float)(sin(a) * (double)mag);
    }
    float ss = 0.0f;
    for (int i = threadIdx.x; i < R; i += 256) ss = fmaf(src[i], src[i], ss);
    ss = block_sum(ss, red);   // (its barriers also publish cs)
    const float inv = 1.0f / sqrtf(ss / (float)R + eps);
    for (int i = threadIdx.x; i < R; i += 256) dst[i] = src[i] * inv * norm_w[i];
    const int pair = halves ? half : 1, step = halves ? 1 : 2;   // pair i = entries (i * step, i * step + pair)
    for (int i = threadIdx.x; i < half; i += 256) {
        float ra, rb;
        rope_rotate(src[R + step * i], src[R + step * i + pair], cs[i], cs[half + i], ra, rb);
        dst[R + step * i] = ra;
        dst[R + step * i + pair] = rb;
    }
    for (int i = dims + threadIdx.x; i < dr; i += 256) dst[R + i] = src[R + i];
    if (q) {
        float* qt = q + (long long)t * ldq;
        for (int j = threadIdx.x; j < H * half; j += 256) {
            const int h = j / half, i = j % half;
            float* p = qt + h * qd + (qd - dr) + step * i;
            float ra, rb;
            rope_rotate(p[0], p[pair], cs[i], cs[half + i], ra, rb);
            p[0] = ra;
            p[pair] = rb;
        }
    }
}

// ------------------------------------------------------------------------------------------------------------------- the attention kernel
struct AttnArgs {
    float* out; int ldo;              // per token
    const float* q; int ldq;          // per token; head h at h * DK
    const float* kA; long long ldA; int nA; int hA;   // first part of a key: kA + (j - keyA0) * ldA + h * hA, nA entries
    const float* kB; long long ldB; int nB;           // second part: kB + j * ldB, nB entries (the rotated part inside the cache row)
    const float* v; long long ldV; int nV; int hV;    // value: v + (j - keyA0) * ldV + h * hV
    int keyA0;
    int H, pos0, T, window;
    float scale;
};

constexpr int QROWS = 16, QPW = 4, KCH = 64, SLAB = 64;

__global__ __launch_bounds__(256) void latent_attention_kernel(const AttnArgs a) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int DK = a.nA + a.nB;
    const int DKP = (DK + 3) & ~3;
    float* Qs = lds;                               // [QROWS][DKP]
    float* Sl = Qs + QROWS * DKP;                  // [KCH][SLAB + 1] key slab / [KCH][SLAB] value slab
    float* Ps = Sl + KCH * (SLAB + 1);             // [QROWS][KCH]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // rows of this workgroup
    const int head = blockIdx.y, n_rows_total = a.T;   // rows = the tokens of this portion, for one head
    const int row0 = blockIdx.x * QROWS;
    auto row_token = [&](int i) { return row0 + i; };
    auto row_head = [&](int) { return head; };
    const int last_row = min(row0 + QROWS, n_rows_total) - 1;
    const int pmin = a.pos0 + row0;
    const int pmax = a.pos0 + last_row;
    const int jlo = a.window > 0 ? max(0, pmin - a.window + 1) : 0;
    const int jhi = pmax;   // inclusive
    // queries into LDS
    for (int d = threadIdx.x; d < DKP; d += 256) {
        float qv[QROWS];
#pragma unroll
        for (int i = 0; i < QROWS; ++i) qv[i] = (row0 + i < n_rows_total && d < DK) ? a.q[(long long)row_token(i) * a.ldq + (long long)row_head(i) * DK + d] : 0.0f;
#pragma unroll
        for (int i = 0; i < QROWS; ++i) Qs[i * DKP + d] = qv[i];
    }
    float m[QPW], l[QPW], acc[QPW][8];
    int rpos[QPW];
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
        m[i] = -INFINITY; l[i] = 0.0f;
        const int ri = wave * QPW + i;
        rpos[i] = row0 + ri < n_rows_total ? a.pos0 + row_token(ri) : -1;
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[i][c] = 0.0f;
    }
    const int hk = head;
    for (int j0 = jlo; j0 <= jhi; j0 += KCH) {
        const int nk = min(KCH, jhi + 1 - j0);
        float s[QPW];
#pragma unroll
        for (int i = 0; i < QPW; ++i) s[i] = 0.0f;
        // ---- scores: slabs of SLAB key entries
        for (int d0 = 0; d0 < DK; d0 += SLAB) {
            const int nd = min(SLAB, DK - d0);
            __syncthreads();
            {   // thread -> (key wave + 4 u, entry lane): the sixteen requests of a thread in flight before the first is stored
                const int d = lane, dd = d0 + d;
                const bool first = dd < a.nA;
                const float* src = first ? a.kA + (long long)(j0 - a.keyA0) * a.ldA + (long long)hk * a.hA + dd : a.kB + (long long)j0 * a.ldB + (dd - a.nA);
                const long long ld = first ? a.ldA : a.ldB;
                float v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    const int k = wave + 4 * u;
                    v[u] = (k < nk && d < nd) ? src[k * ld] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 16; ++u) Sl[(wave + 4 * u) * (SLAB + 1) + d] = v[u];
            }
            __syncthreads();
            const float* kr = Sl + lane * (SLAB + 1);
            for (int d = 0; d < nd; d += 4) {      // (entries past nd are zero in the slab, past DK in the queries)
                const float k0 = kr[d], k1 = kr[d + 1], k2 = kr[d + 2], k3 = kr[d + 3];
#pragma unroll
                for (int i = 0; i < QPW; ++i) {
                    const float4 q4 = *reinterpret_cast<const float4*>(Qs + (wave * QPW + i) * DKP + d0 + d);
                    s[i] = fmaf(q4.x, k0, s[i]); s[i] = fmaf(q4.y, k1, s[i]); s[i] = fmaf(q4.z, k2, s[i]); s[i] = fmaf(q4.w, k3, s[i]);
                }
            }
        }
        // ---- online softmax, weights to LDS
        const int j = j0 + lane;
#pragma unroll
        for (int i = 0; i < QPW; ++i) {
            const bool vis = lane < nk && rpos[i] >= 0 && j <= rpos[i] && (a.window <= 0 || rpos[i] - j < a.window);
            const float sv = vis ? s[i] * a.scale : -INFINITY;
            const float mn = fmaxf(m[i], wave_max(sv));
            const float ms = mn == -INFINITY ? 0.0f : mn;
            const float p = vis ? expf(sv - ms) : 0.0f;
            const float corr = m[i] == -INFINITY ? 0.0f : expf(m[i] - ms);
            l[i] = l[i] * corr + wave_sum(p);
            m[i] = mn;
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[i][c] *= corr;
            Ps[(wave * QPW + i) * KCH + lane] = p;
        }
        // ---- weighted sum: slabs of SLAB value columns, lane = column
        const int hv = head;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int v0 = c * SLAB;
            if (v0 < a.nV) {
                const int nvv = min(SLAB, a.nV - v0);
                __syncthreads();
                {
                    const float* src = a.v + (long long)(j0 - a.keyA0) * a.ldV + (long long)hv * a.hV + v0 + lane;
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int k = wave + 4 * u;
                        v[u] = (k < nk && lane < nvv) ? src[k * a.ldV] : 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) Sl[(wave + 4 * u) * SLAB + lane] = v[u];
                }
                __syncthreads();
                for (int k = 0; k < nk; k += 4) {      // (weights and value rows past nk are zero)
                    const float x0 = Sl[k * SLAB + lane], x1 = Sl[(k + 1) * SLAB + lane], x2 = Sl[(k + 2) * SLAB + lane], x3 = Sl[(k + 3) * SLAB + lane];
#pragma unroll
                    for (int i = 0; i < QPW; ++i) {
                        const float4 p4 = *reinterpret_cast<const float4*>(Ps + (wave * QPW + i) * KCH + k);
                        acc[i][c] = fmaf(p4.x, x0, acc[i][c]); acc[i][c] = fmaf(p4.y, x1, acc[i][c]);
                        acc[i][c] = fmaf(p4.z, x2, acc[i][c]); acc[i][c] = fmaf(p4.w, x3, acc[i][c]);
                    }
                }
            }
        }
    }
    // ---- results
#pragma unroll
    for (int i = 0; i < QPW; ++i) {
        const int ri = wave * QPW + i;
        if (row0 + ri >= n_rows_total) continue;
        const int t = row_token(ri), h = row_head(ri);
        const float inv = l[i] > 0.0f ? 1.0f / l[i] : 0.0f;
        float* o = a.out + (long long)t * a.ldo + (long long)h * a.nV;
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (c * SLAB + lane < a.nV) o[c * SLAB + lane] = acc[i][c] * inv;
    }
}

// ------------------------------------------------------------------------------------------------------------------- the shared form (decoding)
// Keys and values are the cache rows themselves.  A workgroup takes 32 of them (KB) for a tile of 16 (token, head) rows on the F32 matrix instructions, and the operands go from memory
// into registers as they are needed: wave w forms the scores over every NWth step of 16 entries (a lane's four entries of a key, as of its query), the parts meet in LDS,
// NW * 4 threads run the online softmax of a row, then wave w sums columns 64 w ..: a lane's four columns of a key are one request and belong to four tiles of results, so
// its results are four neighbours too.  The tiles of 32 keys go round `splits` workgroups; each leaves one (max, sum) and one vector per row, joined in the launch behind.
// Latency bounds it with few positions: launch, ONE round trip for queries, keys and values together, 40 matrix instructions a wave, softmax, 32 more, the states out.  us, 16 heads,
// 512 + 64, a token at 44 / 1100 positions: four waves with the tile in LDS 11.4 / 13.0, so 8.6 / 9.4; the matrix instructions bound it with many: with the merge, 8000 31.9 -> 19.2, 32000
// 92.7 -> 44.4 (the next tile's rows are on their way under this one's work, and two workgroups fit on a CU).
constexpr int KB = 32, SROWS = 16;
struct SharedArgs {
    const float* q; int ldq;          // [T][H][R + dr], ldq floats between tokens
    const float* cache; int row;      // cache rows
    int R, dr, H, pos0, T, window, splits;
    float scale;
    float* scratch;                   // [rows][splits][R] vectors, then [rows][splits][2] maxima and sums
};

// NW waves: ranks up to 64 * NW; KS: keys of (latent + rotated) up to 16 * NW * KS entries; V: rows of whole fours on 16 bytes.  The smaller sizes need fewer registers, which
// counts where many rows walk a long context.  us with the merge, 8 tokens of 64 heads at 8000 positions, tile in LDS / so: 32 + 8 121 / 43, 256 + 32 157 / 95, 512 + 64 400 / 193.
// ROUTE: the first `beside` rows of the grid's workgroups choose a token's experts each (route_token), which waits for nothing that attention leaves.  Attention of one token leaves most
// CUs idle and takes about as long: us, 16 heads, 512 + 64, 1100 positions, and a router of 32 experts of 2048 inputs: 9.6 + 8.7 in two launches, 10.8 so (12.5 with four rows
// of the router a wave, requested behind the norm).  Five rows a wave are one round for up to 40 rows; with more the launch gains less, but it gains: with the unfolding behind it, two launches / so, 16 .. 39
// experts 1.5, 64 23.8 / 16.5, 128 29.2 / 23.8, 256 39.7 / 35.1; of 4096 inputs 256 57.4 / 56.2; over 1, 2 and 8 tokens at 40, 1100 and 8000 positions 1.00 .. 1.60.
struct NoRoute {};
struct RouteBeside { RouteJob job; int T, rows; };
constexpr int kRouteBesideInputs = 4096;
template <int KS, int NW, bool V, bool ROUTE = false>
__global__ __launch_bounds__(64 * NW) void latent_attention_shared_kernel(const SharedArgs a, const std::conditional_t<ROUTE, RouteBeside, NoRoute> route) {
    int part = blockIdx.y;
    if constexpr (ROUTE) {
        __shared__ __attribute__((aligned(16))) float xs[kRouteBesideInputs];
        if (part < route.rows) {
            const int t = part * (int)gridDim.x + (int)blockIdx.x;
            if (t < route.T) route_token<NW, 5>(route.job, t, xs);
            return;
        }
        part -= route.rows;
    }
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef f4 f4_anywhere __attribute__((aligned(4)));
    constexpr int PP = KB + 4, TPR = 4 * NW, KPT = KB / TPR;       // softmax: threads a row, keys a thread
    __shared__ float Sp[NW * SROWS * PP];          // parts of the scores
    __shared__ __attribute__((aligned(16))) float Ps[SROWS * PP];
    __shared__ float ms[SROWS], ls[SROWS], cr[SROWS];      // running max and sum, correction of this tile
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i16 = lane & 15, g4 = lane >> 4;
    const int DK = a.R + a.dr, steps = (DK + 15) / 16, col = 64 * wave + 4 * i16;
    const int n_rows = a.T * a.H, row0 = blockIdx.x * SROWS;
    const int last_row = min(row0 + SROWS, n_rows) - 1;
    const int pmin = a.pos0 + row0 / a.H, pmax = a.pos0 + last_row / a.H;
    const int jlo = a.window > 0 ? max(0, pmin - a.window + 1) : 0, jhi = pmax;
    // entries at .. at + 3 of a row of `end`, zero behind it: asked for, and what was asked for as it is used.  As they lie (V); else every request goes out unconditionally and what does not count is moved or zeroed
    // when it is used: keys of up to 128 entries one by one, past the end the last one again; longer ones in fours, a row's last entries with the four that end it.  (Requests under conditions were waited
    // for one after the other.  us with merge and unfolding, the tile in LDS / those / so: 9 entries at 172 positions 10.6 / 12.9 / 11.5, 255 + 30 at 128 17.2 / 15.0 / 13.8)
    constexpr bool SINGLE = !V && KS == 2;
    auto ask = [](const float* p, int at, int end) -> f4 {
        f4 v{0.f, 0.f, 0.f, 0.f};
        if constexpr (V) { if (at < end) v = *reinterpret_cast<const f4*>(p + at); }
        else if constexpr (!SINGLE) v = *reinterpret_cast<const f4_anywhere*>(p + min(at, max(end, 4) - 4));          // (end < 4: a rank beside rotated entries, which are four at least together)
        else
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = p[min(at + c, end - 1)];
        return v;
    };
    auto put = [](const f4& w, int at, int end) -> f4 {
        if constexpr (V) return w;
        else if constexpr (SINGLE) return f4{at < end ? w[0] : 0.f, at + 1 < end ? w[1] : 0.f, at + 2 < end ? w[2] : 0.f, at + 3 < end ? w[3] : 0.f};
        const int back = at - min(at, max(end, 4) - 4);                 // (past a rank below four: columns that nothing reads)
        return back == 0 ? w : back == 1 ? f4{w[1], w[2], w[3], 0.f} : back == 2 ? f4{w[2], w[3], 0.f, 0.f} : back == 3 ? f4{w[3], 0.f, 0.f, 0.f} : f4{0.f, 0.f, 0.f, 0.f};
    };
    // (keys past the last re-read it; their weight is zero)
    f4 qf[KS], kf[KS][2], vf[2][4];
    auto load_keys = [&](int j0) {
        const float* k0 = a.cache + (long long)min(j0 + i16, jhi) * a.row, *k1 = a.cache + (long long)min(j0 + 16 + i16, jhi) * a.row;
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            const int st = wave + NW * u;
            if (st < steps) { kf[u][0] = ask(k0, 16 * st + 4 * g4, DK); kf[u][1] = ask(k1, 16 * st + 4 * g4, DK); }
        }
    };
    const bool sums = 64 * wave < a.R;             // (uniform over the wave)
    auto load_values = [&](int j0) {
        if (!sums) return;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int c = 0; c < 4; ++c) vf[e][c] = ask(a.cache + (long long)min(j0 + 16 * e + 4 * g4 + c, jhi) * a.row, col, a.R);
    };
    int j0 = jlo + KB * part;
    const int hop = KB * a.splits;
    {
        const int r = min(row0 + i16, n_rows - 1);
        const float* q = a.q + (long long)(r / a.H) * a.ldq + (long long)(r % a.H) * DK;
#pragma unroll
        for (int u = 0; u < KS; ++u)
            if (wave + NW * u < steps) qf[u] = ask(q, 16 * (wave + NW * u) + 4 * g4, DK);
    }
    if (j0 <= jhi) { load_keys(j0); load_values(j0); }
    if constexpr (!V)
#pragma unroll
        for (int u = 0; u < KS; ++u)
            if (wave + NW * u < steps) qf[u] = put(qf[u], 16 * (wave + NW * u) + 4 * g4, DK);
    if (tid < SROWS) { ms[tid] = -INFINITY; ls[tid] = 0.0f; }
    const int srow = tid / TPR, sub = tid % TPR;
    const int rpos = row0 + srow < n_rows ? a.pos0 + (row0 + srow) / a.H : -1;
    f4 acc[4];                                     // column 64 wave + 4 i16 + t of rows 4 g4 ..
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    for (; j0 <= jhi; j0 += hop) {
        const int nk = min(KB, jhi + 1 - j0);
        const bool more = j0 + hop <= jhi;
        // ---- scores: this wave's steps
        f4 s0{0.f, 0.f, 0.f, 0.f}, s1{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            if (wave + NW * u >= steps) continue;  // (uniform over the wave)
            const int at = 16 * (wave + NW * u) + 4 * g4;
            const f4 k0 = put(kf[u][0], at, DK), k1 = put(kf[u][1], at, DK);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[u][c], k0[c], s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[u][c], k1[c], s1, 0, 0, 0);
            }
        }
        if (more) load_keys(j0 + hop);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            Sp[(wave * SROWS + 4 * g4 + r) * PP + i16] = s0[r];
            Sp[(wave * SROWS + 4 * g4 + r) * PP + 16 + i16] = s1[r];
        }
        __syncthreads();                           // (also: every wave has read the previous tile's weights)
        // ---- online softmax
        {
            float sv[KPT], mc = -INFINITY;
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                const int key = sub + TPR * e, j = j0 + key;
                float sc[NW];
#pragma unroll
                for (int w = 0; w < NW; ++w) sc[w] = Sp[(w * SROWS + srow) * PP + key];
#pragma unroll
                for (int n = NW / 2; n; n >>= 1)
#pragma unroll
                    for (int w = 0; w < n; ++w) sc[w] += sc[w + n];
                const bool vis = key < nk && rpos >= 0 && j <= rpos && (a.window <= 0 || rpos - j < a.window);
                sv[e] = vis ? sc[0] * a.scale : -INFINITY;
                mc = fmaxf(mc, sv[e]);
            }
#pragma unroll
            for (int o = TPR / 2; o >= 1; o >>= 1) mc = fmaxf(mc, __shfl_xor(mc, o, TPR));
            const float mo = ms[srow];
            const float mn = fmaxf(mo, mc), msafe = mn == -INFINITY ? 0.0f : mn;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                const float p = sv[e] == -INFINITY ? 0.0f : expf(sv[e] - msafe);
                Ps[srow * PP + sub + TPR * e] = p;
                sum += p;
            }
#pragma unroll
            for (int o = TPR / 2; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, TPR);
            if (sub == 0) {                        // (the row's lanes are of one wave: all have read ms)
                const float corr = mo == -INFINITY ? 0.0f : expf(mo - msafe);
                ls[srow] = ls[srow] * corr + sum;
                ms[srow] = mn;
                cr[srow] = corr;
            }
        }
        __syncthreads();
        // ---- weighted latents: this wave's columns
        if (sums) {
            const f4 p0 = *reinterpret_cast<const f4*>(&Ps[i16 * PP + 4 * g4]), p1 = *reinterpret_cast<const f4*>(&Ps[i16 * PP + 16 + 4 * g4]);
            float corr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) corr[r] = cr[4 * g4 + r];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][r] *= corr[r];
#pragma unroll
            for (int c = 0; c < 4; ++c) {          // component c of the weights belongs to key 4 g4 + c
                const f4 v0 = put(vf[0][c], col, a.R), v1 = put(vf[1][c], col, a.R);
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p0[c], v0[t], acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p1[c], v1[t], acc[t], 0, 0, 0);
                }
            }
            if (more) load_values(j0 + hop);
        }
    }
    __syncthreads();                               // (a workgroup without a tile: ms is written)
    const long long states = (long long)n_rows * a.splits;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 4 * g4 + r;
        if (row0 + i >= n_rows) continue;
        const long long at = (long long)(row0 + i) * a.splits + part;
        if (wave == 0 && i16 == 0) { a.scratch[states * a.R + 2 * at] = ms[i]; a.scratch[states * a.R + 2 * at + 1] = ls[i]; }
        float* st = a.scratch + at * a.R;
        if constexpr (V) { if (col < a.R) *reinterpret_cast<f4*>(st + col) = f4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]}; }
        else
#pragma unroll
            for (int t = 0; t < 4; ++t) if (col + t < a.R) st[col + t] = acc[t][r];
    }
}

// merge of the partial states of one (token, head) row: weights of the states first, then a workgroup sums 64 columns over them, a quarter of the states per wave (one
// workgroup per row walked all columns over all states: 7.0 us at 35 states of 512, 4.1 this way)
__global__ __launch_bounds__(256) void latent_attention_merge_kernel(float* out, int ldo, const float* scratch, int splits, int nV, int H) {
    __shared__ float wt[256];
    __shared__ float red[16];
    __shared__ float part[4][64];
    const int r = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;   // r = t * H + h
    const float* st = scratch + (long long)r * splits * nV, *ml = scratch + ((long long)gridDim.x * nV + 2LL * r) * splits;
    const long long step = nV;
    const int v = blockIdx.y * 64 + lane, each = (splits + 3) / 4, s0 = wave * each, s1 = min(s0 + each, splits);
    float x[8];                                    // the wave's first eight states requested together with the maxima
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = s0 + u < s1 && v < nV ? st[(s0 + u) * step + v] : 0.0f;
    const int mine = threadIdx.x;                  // (at most 128 states)
    const float m = mine < splits ? ml[2 * mine] : -INFINITY, l = mine < splits ? ml[2 * mine + 1] : 0.0f;
    const float mx = block_max(m, red);
    const float w = m == -INFINITY ? 0.0f : expf(m - mx);
    wt[threadIdx.x] = w;
    const float den = block_sum(w * l, red);       // (its barriers publish wt)
    const float inv = den > 0.0f ? 1.0f / den : 0.0f;
    float sum = 0.0f;
    for (int s = s0; s < s1; s += 8) {             // states in order
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s + u < s1) sum = fmaf(x[u], wt[s + u], sum);
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = s + 8 + u < s1 && v < nV ? st[(s + 8 + u) * step + v] : 0.0f;
    }
    part[wave][lane] = sum;
    __syncthreads();
    if (wave == 0 && v < nV) out[(long long)(r / H) * ldo + (long long)(r % H) * nV + v] = ((part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane])) * inv;
}

// ------------------------------------------------------------------------------------------------------------------- fold / unfold
// qf[t][h][r] = sum_d q[t][h][d] W_uk[h * dn + d][r]; rotated part copied behind.  grid (R / 64, H, T): 64 columns per workgroup, the d range in
// four parts (one per wave), added through LDS in wave order
// kv != NULL: the workgroups (0, H, T) write the tokens' cache rows beside that -- normed latents, rotated key parts -- and the queries' rotated parts turn on their way (dr == 0: neither has
// one), by latent_prepare_kernel's expressions.  A decoded token's two launches of 5.0 and 4.2 us are one of 4.6 - 4.9 (16 heads of 128 + 64, rank 512).
struct FoldPrepare { float* cache; int row; const float* kv; int ldkv; const float* norm_w; float eps; int pos0; const double* freq; float mag; int dims, halves; };
template <typename WT>
__global__ __launch_bounds__(256) void latent_fold_query_kernel(float* qf, const float* q, int ldq, const WT* w, int H, int dn, int dr, int R, const FoldPrepare p) {
    extern __shared__ float qs[];      // [dn + dr] then [4][64] partial sums
    if ((int)blockIdx.y == H) {        // (uniform over the workgroup)
        if (blockIdx.x > 0) return;
        const float* src = p.kv + (long long)blockIdx.z * p.ldkv;
        float* dst = p.cache + (long long)(p.pos0 + blockIdx.z) * p.row;
        float ss = 0.0f;
        for (int i = threadIdx.x; i < R; i += 256) ss = fmaf(src[i], src[i], ss);
        const float inv = 1.0f / sqrtf(block_sum(ss, qs) / (float)R + p.eps);
        for (int i = threadIdx.x; i < R; i += 256) dst[i] = src[i] * inv * p.norm_w[i];
        const int half = p.dims / 2, pair = p.halves ? half : 1, step = p.halves ? 1 : 2;
        for (int i = threadIdx.x; i < half; i += 256) {
            const double ang = (double)(p.pos0 + (int)blockIdx.z) * p.freq[i];
            float ra, rb;
            rope_rotate(src[R + step * i], src[R + step * i + pair], (float)(cos(ang) * (double)p.mag), (float)(sin(ang) * (double)p.mag), ra, rb);
            dst[R + step * i] = ra;
            dst[R + step * i + pair] = rb;
        }
        for (int i = p.dims + threadIdx.x; i < dr; i += 256) dst[R + i] = src[R + i];
        return;
    }
    float* part = qs + dn + dr;
    const int h = blockIdx.y, t = blockIdx.z;
    const float* qh = q + (long long)t * ldq + (long long)h * (dn + dr);
    float* o = qf + ((long long)t * H + h) * (R + dr);
    for (int d = threadIdx.x; d < dn + dr; d += 256) qs[d] = qh[d];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = blockIdx.x * 64 + lane;
    const int per = (dn + 3) / 4, d0 = wave * per, d1 = min(d0 + per, dn);
    const WT* wh = w + (long long)h * dn * R;
    float s = 0.0f;
    if (r < R) {
#pragma unroll 8
        for (int d = d0; d < d1; ++d) {
            float wv;
            if constexpr (sizeof(WT) == 2) wv = __uint_as_float((uint32_t)wh[(long long)d * R + r] << 16); else wv = wh[(long long)d * R + r];
            s = fmaf(qs[d], wv, s);
        }
    }
    part[wave * 64 + lane] = s;
    __syncthreads();
    if (wave == 0 && r < R) o[r] = ((part[lane] + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
    if (blockIdx.x == 0) {
        const int half = p.dims / 2, pair = p.halves ? half : 1, step = p.halves ? 1 : 2;
        for (int i = threadIdx.x; i < half; i += 256) {
            const double ang = (double)(p.pos0 + t) * p.freq[i];
            float ra, rb;
            rope_rotate(qs[dn + step * i], qs[dn + step * i + pair], (float)(cos(ang) * (double)p.mag), (float)(sin(ang) * (double)p.mag), ra, rb);
            o[R + step * i] = ra;
            o[R + step * i + pair] = rb;
        }
        for (int d = p.dims + threadIdx.x; d < dr; d += 256) o[R + d] = qs[dn + d];
    }
}

// out[t][h * dv + v] = W_uv[h * dv + v][:] . lat[t][h][:] (* sigmoid(gate));  grid (dv / 16, H, T): a wave owns 4 outputs and walks their rows together
template <typename WT>
__global__ __launch_bounds__(256) void latent_unfold_value_kernel(float* out, int ldo, const float* lat, const WT* w, const float* gate, int ldg, int H, int dv,
                                                                 int R, int head_gate) {
    extern __shared__ float ls[];
    const int h = blockIdx.y, t = blockIdx.z;
    const float* lh = lat + ((long long)t * H + h) * R;
    for (int r = threadIdx.x; r < R; r += 256) ls[r] = lh[r];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v0 = blockIdx.x * 16 + wave * 4;
    if (v0 >= dv) return;
    const WT* wr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wr[i] = w + ((long long)h * dv + min(v0 + i, dv - 1)) * R;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int r = lane; r < R; r += 64) {
        float wv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (sizeof(WT) == 2) wv[i] = __uint_as_float((uint32_t)wr[i][r] << 16); else wv[i] = wr[i][r];
        }
        const float x = ls[r];
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = fmaf(wv[i], x, s[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float tsum = wave_sum_lane63(s[i]);
        if (lane == 63 && v0 + i < dv) {
            if (gate) tsum *= 1.0f / (1.0f + expf(-gate[(long long)t * ldg + (head_gate ? h : h * dv + v0 + i)]));
            out[(long long)t * ldo + h * dv + v0 + i] = tsum;
        }
    }
}

// ... with the parts' states (latent_attention_shared_kernel) joined in front, for ranks of whole pieces of eight up to 512: every workgroup of a head joins them for itself.  All
// states are requested at once with the matrix rows: a thread takes four columns of every fourth state, the four parts of a column meet in LDS; a wave then owns four outputs.
// us of the merge above and the unfolding / with the states eight after eight and 16 outputs a workgroup / so, 16 heads of 128, rank 512, one token: 2 states 3.6 + 6.0 / 5.1 / 4.9, 36 states
// 4.1 + 6.4 / 8.3 / 5.2
constexpr int kJoinStates = 48;                          // (states of all tokens: beyond, what the workgroups of a head read again costs more than the launch)
template <typename WT>
__global__ __launch_bounds__(512) void latent_join_unfold_kernel(float* out, int ldo, const float* scratch, int splits, const WT* w, const float* gate, int ldg, int H, int dv, int R, int head_gate) {
    constexpr int EACH = kJoinStates / 4;
    __shared__ float wt[kJoinStates], red;
    __shared__ __attribute__((aligned(16))) float part[4][512];
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int h = blockIdx.y, t = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int v0 = blockIdx.x * 32 + wave * 4, r0 = lane * 8, c = 4 * (tid & 127), mine = tid >> 7;
    const long long at = ((long long)t * H + h) * splits, states = (long long)gridDim.z * H * splits;
    const float* st = scratch + at * R, *ml = scratch + states * R + 2 * at;
    float m = -INFINITY, l = 0.0f;
    if (wave == 0 && lane < splits) { m = ml[2 * lane]; l = ml[2 * lane + 1]; }
    f4 x[EACH];
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
        x[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        if (4 * u + mine < splits && c < R) x[u] = *reinterpret_cast<const f4*>(st + (long long)(4 * u + mine) * R + c);
    }
    float wv[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const WT* row = w + ((long long)h * dv + min(v0 + i, dv - 1)) * R + r0;
        if constexpr (sizeof(WT) == 2) {
            uint4 b{0u, 0u, 0u, 0u};
            if (r0 < R) b = *reinterpret_cast<const uint4*>(row);
            const uint32_t u[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) { wv[i][2 * k] = __uint_as_float(u[k] << 16); wv[i][2 * k + 1] = __uint_as_float(u[k] & 0xFFFF0000u); }
        } else {
            float4 a{0.0f, 0.0f, 0.0f, 0.0f}, b = a;
            if (r0 < R) { a = *reinterpret_cast<const float4*>(row); b = *reinterpret_cast<const float4*>(row + 4); }
            wv[i][0] = a.x; wv[i][1] = a.y; wv[i][2] = a.z; wv[i][3] = a.w; wv[i][4] = b.x; wv[i][5] = b.y; wv[i][6] = b.z; wv[i][7] = b.w;
        }
    }
    if (wave == 0) {                                     // (at most 48 states: one wave has them)
        const float mx = wave_max(m);
        const float we = m == -INFINITY ? 0.0f : expf(m - mx);
        if (lane < kJoinStates) wt[lane] = we;           // (zero behind the last)
        const float den = wave_sum(we * l);
        if (lane == 0) red = den > 0.0f ? 1.0f / den : 0.0f;
    }
    __syncthreads();
    f4 sum{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < EACH; ++u) {
        const float we = wt[4 * u + mine];
#pragma unroll
        for (int k = 0; k < 4; ++k) sum[k] = fmaf(x[u][k], we, sum[k]);
    }
    *reinterpret_cast<f4*>(&part[mine][c]) = sum;
    __syncthreads();
    if (v0 >= dv) return;
    const float inv = red;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (r0 < R) {
        float xx[8];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const f4 p0 = *reinterpret_cast<const f4*>(&part[0][r0 + 4 * k]), p1 = *reinterpret_cast<const f4*>(&part[1][r0 + 4 * k]), p2 = *reinterpret_cast<const f4*>(&part[2][r0 + 4 * k]),
                     p3 = *reinterpret_cast<const f4*>(&part[3][r0 + 4 * k]);
#pragma unroll
            for (int j = 0; j < 4; ++j) xx[4 * k + j] = ((p0[j] + p1[j]) + (p2[j] + p3[j])) * inv;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int k = 0; k < 8; ++k) s[i] = fmaf(wv[i][k], xx[k], s[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float tsum = wave_sum_lane63(s[i]);
        if (lane == 63 && v0 + i < dv) {
            if (gate) tsum *= 1.0f / (1.0f + expf(-gate[(long long)t * ldg + (head_gate ? h : h * dv + v0 + i)]));
            out[(long long)t * ldo + h * dv + v0 + i] = tsum;
        }
    }
}

static int shared_splits(int nkeys) {       // workgroups per row tile: one per tile of KB keys, at most 128
    const int tiles = (nkeys + KB - 1) / KB + 1;     // (+ 1: a tile's first key is the window's, not a multiple of KB)
    return tiles < 1 ? 1 : tiles > 128 ? 128 : tiles;
}

static int shared_keys(int pos0, int T, int window) { return window > 0 ? (window + T - 1 < pos0 + T ? window + T - 1 : pos0 + T) : pos0 + T; }
static bool shared_whole(const float* q, int ldq, const float* cache, int row, int kv_rank, int rot_dim, const float* scratch) {
    return !((kv_rank | rot_dim | row | ldq) & 3) && !(((uintptr_t)cache | (uintptr_t)q | (uintptr_t)scratch) & 15);
}
// A router beside attention: where the workgroups are of eight waves (four walk the router's rows alone for longer than such attention takes) and a row fits beside a tile.
static bool shared_takes_route(bool whole, int kv_rank, int rot_dim, int n) {
    return whole && kv_rank + rot_dim > 128 && (kv_rank + rot_dim > 320 || kv_rank > 256) && ntk_latent_shared_takes(kv_rank, rot_dim) && n <= kRouteBesideInputs;
}
// the shared form: every part's states into the scratch; merge: joined in `out`
static int launch_shared(SharedArgs& sa, float* out, int ldo, const float* q, int ldq, const float* cache, int row, int kv_rank, int rot_dim, int H, int pos0, int T, int window, float scale,
                         float* scratch, bool merge, void* stream, const RouteBeside* route = nullptr) {
    if (!scratch) return NTK_E_NULL;
    if (!ntk_latent_shared_takes(kv_rank, rot_dim)) return NTK_E_SHAPE;
    hipStream_t s = resolve_stream(stream);
    sa.q = q; sa.ldq = ldq; sa.cache = cache; sa.row = row; sa.R = kv_rank; sa.dr = rot_dim; sa.H = H; sa.pos0 = pos0; sa.T = T; sa.window = window;
    sa.scale = scale; sa.scratch = scratch;
    sa.splits = shared_splits(shared_keys(pos0, T, window));
    const int rows = T * H, DK = kv_rank + rot_dim;
    dim3 grid((rows + SROWS - 1) / SROWS, sa.splits);
    const bool whole = shared_whole(q, ldq, cache, row, kv_rank, rot_dim, scratch);
    auto launch = [&](auto kernel, auto narrow, int waves) {
        if (whole) hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, s, sa, NoRoute{});
        else hipLaunchKernelGGL(narrow, grid, dim3(64 * waves), 0, s, sa, NoRoute{});
    };
    if (route) {                                   // (shared_takes_route)
        RouteBeside r = *route;
        r.rows = (r.T + (int)grid.x - 1) / (int)grid.x;
        grid.y += r.rows;
        if (DK <= 640) hipLaunchKernelGGL((latent_attention_shared_kernel<5, 8, true, true>), grid, dim3(512), 0, s, sa, r);
        else hipLaunchKernelGGL((latent_attention_shared_kernel<7, 8, true, true>), grid, dim3(512), 0, s, sa, r);
    } else
    if (DK <= 128) launch(latent_attention_shared_kernel<2, 4, true>, latent_attention_shared_kernel<2, 4, false>, 4);
    else if (DK <= 320 && kv_rank <= 256) launch(latent_attention_shared_kernel<5, 4, true>, latent_attention_shared_kernel<5, 4, false>, 4);
    else if (DK <= 640) launch(latent_attention_shared_kernel<5, 8, true>, latent_attention_shared_kernel<5, 8, false>, 8);
    else launch(latent_attention_shared_kernel<7, 8, true>, latent_attention_shared_kernel<7, 8, false>, 8);
    const int st = last_launch_status();
    if (st != NTK_OK || !merge) return st;
    hipLaunchKernelGGL(latent_attention_merge_kernel, dim3(rows, (kv_rank + 63) / 64), dim3(256), 0, s, out, ldo, (const float*)scratch, sa.splits, kv_rank, H);
    return last_launch_status();
}

}  // namespace ntk

using namespace ntk;

int ntk_latent_shared_takes(int kv_rank, int rot_dim) {
    return kv_rank > 0 && kv_rank <= 512 && rot_dim >= 0 && kv_rank + rot_dim <= 816;
}

int ntk_latent_prepare(float* cache, int row, const float* kv, int ldkv, const float* norm_w, float eps, int kv_rank, int rot_dim, float* q, int ldq, int H, int qd,
                       const ntk_rotary* rot, int pos0, int T, void* stream) {
    static const ntk_rotary none{nullptr, 1.0f, 0, NTK_ROT_NEIGHBOURS};
    if (!rot) rot = &none;
    if (!cache || !kv || !norm_w || (rot->dims > 0 && !rot->freq)) return NTK_E_NULL;
    if (T < 0 || kv_rank <= 0 || rot_dim < 0 || rot->dims < 0 || (rot->dims & 1) || rot->dims > rot_dim || row < kv_rank + rot_dim || ldkv < kv_rank + rot_dim || pos0 < 0) return NTK_E_SHAPE;
    if (q && (H <= 0 || qd < rot_dim || ldq < H * qd)) return NTK_E_SHAPE;
    if (rot->layout != NTK_ROT_NEIGHBOURS && rot->layout != NTK_ROT_HALVES) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(latent_prepare_kernel, dim3(T), dim3(256), (size_t)(rot_dim + 2) * sizeof(float), resolve_stream(stream), cache, row, kv, ldkv, norm_w,
                       eps, kv_rank, rot_dim, q, ldq, H, qd, rot->freq, rot->mag, rot->dims, pos0, rot->layout == NTK_ROT_HALVES ? 1 : 0);
    return last_launch_status();
}

size_t ntk_latent_attention_scratch(int T, int H, int vdim_or_rank, int nkeys) {
    return (size_t)T * H * shared_splits(nkeys) * (2 + vdim_or_rank);
}

size_t ntk_prompt_attention_image_bytes(int positions, int kv_heads, int key_entries, int value_entries) {
    return positions > 0 && kv_heads > 0 && key_entries > 0 && value_entries > 0 ? piece_attention_bytes((positions - 1) / 32 + 3, kv_heads, key_entries, value_entries) : 0;
}

int ntk_latent_attention(float* out, int ldo, const float* q, int ldq, const float* K, int ldk, const float* V, int ldv, const float* cache, int row,
                         int kv_rank, int rot_dim, int H, int dn, int dv, int shared, int pos0, int T, int key0, int window, float scale, float* scratch,
                         void* stream) {
    return ntk_latent_attention_ex(out, ldo, q, ldq, K, ldk, V, ldv, cache, row, kv_rank, rot_dim, H, dn, dv, shared, pos0, T, key0, window, scale, scratch, nullptr, 0, stream);
}

int ntk_latent_attention_ex(float* out, int ldo, const float* q, int ldq, const float* K, int ldk, const float* V, int ldv, const float* cache, int row,
                            int kv_rank, int rot_dim, int H, int dn, int dv, int shared, int pos0, int T, int key0, int window, float scale, float* scratch,
                            void* image, size_t image_bytes, void* stream) {
    if (!out || !q || !cache) return NTK_E_NULL;
    if (!shared && (!K || !V)) return NTK_E_NULL;
    if (T < 0 || H <= 0 || kv_rank <= 0 || rot_dim < 0 || pos0 < 0 || key0 < 0 || row < kv_rank + rot_dim) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipStream_t s = resolve_stream(stream);
    if (shared) {
        SharedArgs sa{};
        return launch_shared(sa, out, ldo, q, ldq, cache, row, kv_rank, rot_dim, H, pos0, T, window, scale, scratch, true, stream);
    }
    if (dn <= 0 || dv <= 0) return NTK_E_SHAPE;
    AttnArgs a{};
    a.out = out; a.ldo = ldo; a.q = q; a.ldq = ldq;
    a.kB = cache + kv_rank; a.ldB = row; a.nB = rot_dim;
    a.H = H; a.pos0 = pos0; a.T = T; a.window = window; a.scale = scale;
    a.kA = K; a.ldA = ldk; a.nA = dn; a.hA = dn;
    a.v = V; a.ldV = ldv; a.nV = dv; a.hV = dv;
    a.keyA0 = key0;
    const int rows = T;
    if (a.nV > 8 * SLAB) return NTK_E_SHAPE;
    if (rows >= 32 && attention_tile_takes(a.nA + a.nB, a.nV)) {       // (fewer rows leave most of a tile of 32 empty)
        TileAttnArgs t{};
        t.out = out; t.ldo = ldo; t.q = q; t.ldq = ldq; t.kA = a.kA; t.ldA = a.ldA; t.nA = a.nA; t.hA = a.hA; t.kB = a.kB; t.ldB = a.ldB; t.nB = a.nB;
        t.v = a.v; t.ldV = a.ldV; t.nV = a.nV; t.hV = a.hV; t.key0 = key0; t.H = H; t.G = H; t.pos0 = pos0; t.T = T; t.window = window; t.scale = scale; t.out_scale = 1.0f;
        if (!launch_attention_pieces(t, image, image_bytes, s)) launch_attention_tile(t, s);
        return last_launch_status();
    }
    const int DKP = (a.nA + a.nB + 3) & ~3;
    const size_t lds = ((size_t)QROWS * DKP + KCH * (SLAB + 1) + QROWS * KCH) * sizeof(float);
    if (lds > 150 * 1024) return NTK_E_SHAPE;
    const dim3 grid((rows + QROWS - 1) / QROWS, H, 1);
    if (lds > 48 * 1024) {
        static bool raised = false;   // (idempotent: a race sets the same attribute twice)
        if (!raised) { NTK_HIP_TRY(hipFuncSetAttribute((const void*)latent_attention_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024)); raised = true; }
    }
    hipLaunchKernelGGL(latent_attention_kernel, grid, dim3(256), lds, s, a);
    return last_launch_status();
}

static int fold_query(float* qf, const float* q, int ldq, const void* w_uk, int wdtype, int T, int H, int dn, int dr, int R, const FoldPrepare& p, void* stream) {
    if (!qf || !q || !w_uk) return NTK_E_NULL;
    if (T < 0 || H <= 0 || dn <= 0 || dr < 0 || R <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const size_t lds = (size_t)(dn + dr + 256) * sizeof(float);
    const dim3 grid((R + 63) / 64, H + (p.kv ? 1 : 0), T);
    if (wdtype == NTK_DT_BF16) hipLaunchKernelGGL(latent_fold_query_kernel<uint16_t>, grid, dim3(256), lds, resolve_stream(stream), qf, q, ldq, (const uint16_t*)w_uk, H, dn, dr, R, p);
    else if (wdtype == NTK_DT_F32) hipLaunchKernelGGL(latent_fold_query_kernel<float>, grid, dim3(256), lds, resolve_stream(stream), qf, q, ldq, (const float*)w_uk, H, dn, dr, R, p);
    else return NTK_E_DTYPE;
    return last_launch_status();
}

int ntk_latent_fold_query(float* qf, const float* q, int ldq, const void* w_uk, int wdtype, int T, int H, int dn, int dr, int R, void* stream) {
    return fold_query(qf, q, ldq, w_uk, wdtype, T, H, dn, dr, R, FoldPrepare{}, stream);
}

int ntk_latent_fold_query_rotate(float* qf, const float* q, int ldq, const void* w_uk, int wdtype, int T, int H, int dn, int dr, int R, const ntk_rotary* rot, float* cache, int row,
                                 const float* kv, int ldkv, const float* norm_w, float eps, int pos0, void* stream) {
    if (!cache || !kv || !norm_w || !rot || (rot->dims > 0 && !rot->freq)) return NTK_E_NULL;
    if (dr < 0 || rot->dims < 0 || (rot->dims & 1) || rot->dims > dr || row < R + dr || ldkv < R + dr || pos0 < 0) return NTK_E_SHAPE;
    if (rot->layout != NTK_ROT_NEIGHBOURS && rot->layout != NTK_ROT_HALVES) return NTK_E_SHAPE;
    return fold_query(qf, q, ldq, w_uk, wdtype, T, H, dn, dr, R, FoldPrepare{cache, row, kv, ldkv, norm_w, eps, pos0, rot->freq, rot->mag, rot->dims, rot->layout == NTK_ROT_HALVES ? 1 : 0}, stream);
}

int ntk_latent_fold_query_prepare(float* qf, const float* q, int ldq, const void* w_uk, int wdtype, int T, int H, int dn, int R, float* cache, int row, const float* kv,
                                  int ldkv, const float* norm_w, float eps, int pos0, void* stream) {
    const ntk_rotary none{nullptr, 1.0f, 0, NTK_ROT_NEIGHBOURS};
    return ntk_latent_fold_query_rotate(qf, q, ldq, w_uk, wdtype, T, H, dn, 0, R, &none, cache, row, kv, ldkv, norm_w, eps, pos0, stream);
}

int ntk_latent_attention_unfold(float* out, int ldo, const void* w_uv, int wdtype, const float* gate, int ldg, int head_gate, int dv, float* lat, const float* qf, const float* cache, int row,
                                int kv_rank, int rot_dim, int H, int pos0, int T, int window, float scale, float* scratch, void* stream) {
    return ntk_latent_attention_unfold_route(out, ldo, w_uv, wdtype, gate, ldg, head_gate, dv, lat, qf, cache, row, kv_rank, rot_dim, H, pos0, T, window, scale, scratch, nullptr, stream);
}

int ntk_latent_attention_unfold_route(float* out, int ldo, const void* w_uv, int wdtype, const float* gate, int ldg, int head_gate, int dv, float* lat, const float* qf, const float* cache, int row,
                                      int kv_rank, int rot_dim, int H, int pos0, int T, int window, float scale, float* scratch, const ntk_norm_route* route, void* stream) {
    if (!out || !w_uv || !lat || !qf || !cache || !scratch) return NTK_E_NULL;
    if (wdtype != NTK_DT_BF16 && wdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (T < 0 || H <= 0 || dv <= 0 || kv_rank <= 0 || rot_dim < 0 || pos0 < 0 || row < kv_rank + rot_dim) return NTK_E_SHAPE;
    RouteBeside rb{};
    if (route) {
        const int st = norm_route_job(route, &rb.job);
        if (st != NTK_OK) return st;
        rb.T = route->T;
    }
    const int ldq = H * (kv_rank + rot_dim);
    const bool beside = route && T > 0 && shared_takes_route(shared_whole(qf, ldq, cache, row, kv_rank, rot_dim, scratch), kv_rank, rot_dim, route->n);
    if (route && !beside) {
        const int st = ntk_moe_norm_route(route->ids, route->wts, route->sgate, route->h, route->ldh, route->x, route->ldx, route->norm_w, route->norm_eps, route->norm_offset, route->w_router,
                                          route->shared_gate_w, route->T, route->n, route->E, route->top, route->form, stream);
        if (st != NTK_OK) return st;
    }
    if (T == 0) return NTK_OK;
    SharedArgs sa{};
    const bool join = kv_rank % 8 == 0 && kv_rank <= 512 && T * shared_splits(shared_keys(pos0, T, window)) <= kJoinStates && !(((uintptr_t)w_uv | (uintptr_t)scratch) & 15);
    const int st = launch_shared(sa, lat, H * kv_rank, qf, ldq, cache, row, kv_rank, rot_dim, H, pos0, T, window, scale, scratch, !join, stream, beside ? &rb : nullptr);
    if (st != NTK_OK) return st;
    if (!join) return ntk_latent_unfold_value_ex(out, ldo, lat, w_uv, wdtype, gate, ldg, head_gate, T, H, dv, kv_rank, stream);
    const dim3 grid((dv + 31) / 32, H, T);
    if (wdtype == NTK_DT_BF16)
        hipLaunchKernelGGL(latent_join_unfold_kernel<uint16_t>, grid, dim3(512), 0, resolve_stream(stream), out, ldo, (const float*)scratch, sa.splits, (const uint16_t*)w_uv, gate, ldg, H, dv, kv_rank, head_gate);
    else
        hipLaunchKernelGGL(latent_join_unfold_kernel<float>, grid, dim3(512), 0, resolve_stream(stream), out, ldo, (const float*)scratch, sa.splits, (const float*)w_uv, gate, ldg, H, dv, kv_rank, head_gate);
    return last_launch_status();
}

int ntk_latent_unfold_value(float* out, int ldo, const float* lat, const void* w_uv, int wdtype, const float* gate, int ldg, int T, int H, int dv, int R,
                            void* stream) {
    return ntk_latent_unfold_value_ex(out, ldo, lat, w_uv, wdtype, gate, ldg, 0, T, H, dv, R, stream);
}

int ntk_latent_unfold_value_ex(float* out, int ldo, const float* lat, const void* w_uv, int wdtype, const float* gate, int ldg, int head_gate, int T, int H, int dv,
                               int R, void* stream) {
    if (!out || !lat || !w_uv) return NTK_E_NULL;
    if (T < 0 || H <= 0 || dv <= 0 || R <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const size_t lds = (size_t)R * sizeof(float);
    const dim3 grid((dv + 15) / 16, H, T);
    if (wdtype == NTK_DT_BF16) hipLaunchKernelGGL(latent_unfold_value_kernel<uint16_t>, grid, dim3(256), lds, resolve_stream(stream), out, ldo, lat, (const uint16_t*)w_uv, gate, ldg, H, dv, R, head_gate);
    else if (wdtype == NTK_DT_F32) hipLaunchKernelGGL(latent_unfold_value_kernel<float>, grid, dim3(256), lds, resolve_stream(stream), out, ldo, lat, (const float*)w_uv, gate, ldg, H, dv, R, head_gate);
    else return NTK_E_DTYPE;
    return last_launch_status();
}
