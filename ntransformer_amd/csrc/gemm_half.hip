// gemm_half.hip -- prompt projections over unquantised GGUF weights (F16): Y[t] (+)= W . X[t] for the tokens of a prompt in one pass over W.
// Replaces, for a prompt, the reference's loop of one GEMV per token (attention.cu / ffn.cpp through gemm.cu:32-470): 200 tokens read the weights 200 times, 18 ms a
// layer of an 8B-shaped F16 model against 0.47 ms as tiles (gemm_tile.hip.h); a 200-token pass of eight such layers 144.5 -> 4.1 ms, 2.9 with the activations' halves formed once and gate | up as one product.  Taken from two tokens on: 16 tokens
// through a 4096 x 4096 matrix take 15 us, one token's GEMV 12.  Products on v_mfma_f32_16x16x32_f16; a 32-bit activation goes in as two halves after
// a per-token power of two (largest |x| in [2^14, 2^15)), which is off by at most 2^-23 of the value (a quarter of them by more than 2^-24, where the one-token
// products take all 24 bits), or by 2^-39 of the row's largest where the second half is subnormal.  The sums make up for it (gemm_tile.hip.h): from
// 3072 inputs on a result is as close to 64 bits as the one-token products' (below, those are closer: 2048 inputs 1.22e-7 of the result against 1.10 .. 1.31e-7, 1024 0.98e-7 against 1.04 .. 1.19e-7).
#include <algorithm>
#include "gemm_direct.hip.h"

namespace ntk {

// largest |x| of every token, one workgroup each (for inputs whose producer has not left it)
__global__ __launch_bounds__(256) void token_max_kernel(float* out, const float* X, int K) {
    __shared__ float red[16];
    const float* x = X + (long long)blockIdx.x * K;
    float m = 0.0f;
    for (int k = threadIdx.x; k < K; k += 256) m = fmaxf(m, fabsf(x[k]));
    m = block_max(m, red);
    if (threadIdx.x == 0) out[blockIdx.x] = m;
}

// The two halves of every activation, planes [2][T][K] (K a multiple of eight), and the rows' largest |x| where their producer has not left them; one workgroup a row.
// In the place of forming them again in each of a product's up to 112 column tiles: 200 rows of 4096 or 14336 in 5.1 .. 5.6 us, with or without the rows' maxima given (a gated unit that
// left them by atomics, four waves a row in each of 112 column tiles, took 192 us in the place of 120).
constexpr float kSplitUs = 4.0f, kSplitRate = 4e6f, kTileUs = 8.0f;     // that launch: us, and bytes per us (eight an entry); what the tiles over 32-bit activations take beside their chunks
constexpr int kHalfKeep = 7;      // pieces of eight a thread keeps (rows up to 14336 cross memory once)
template <bool GIVEN>
__global__ __launch_bounds__(256) void half_split_kernel(_Float16* out, long long plane, const float* X, int K, float* row_max) {
    __shared__ float red[16];
    const float* x = X + (long long)blockIdx.x * K;
    uint16_t* o = reinterpret_cast<uint16_t*>(out) + (long long)blockIdx.x * K;
    float4 v[kHalfKeep][2];
#pragma unroll
    for (int p = 0; p < kHalfKeep; ++p) {
        const int k = 8 * (threadIdx.x + 256 * p);
        v[p][0] = k < K ? *reinterpret_cast<const float4*>(x + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        v[p][1] = k < K ? *reinterpret_cast<const float4*>(x + k + 4) : float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float largest;
    if constexpr (GIVEN) largest = row_max[blockIdx.x];
    else {
        float m = 0.0f;
#pragma unroll
        for (int p = 0; p < kHalfKeep; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q) m = fmaxf(fmaxf(fmaxf(m, fabsf(v[p][q].x)), fmaxf(fabsf(v[p][q].y), fabsf(v[p][q].z))), fabsf(v[p][q].w));
        for (int k = 8 * (threadIdx.x + 256 * kHalfKeep); k < K; k += 8 * 256)
#pragma unroll
            for (int j = 0; j < 8; ++j) m = fmaxf(m, fabsf(x[k + j]));
        largest = block_max(m, red);
        if (threadIdx.x == 0) row_max[blockIdx.x] = largest;
    }
    const float scale = half_scale(largest);
    auto put = [&](int k, const float4 a, const float4 b) {
        const float e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uintx4_t u[2];
        TileHalf2::convert(e, scale, u);
        *reinterpret_cast<uintx4_t*>(o + k) = u[0];
        *reinterpret_cast<uintx4_t*>(o + plane + k) = u[1];
    };
#pragma unroll
    for (int p = 0; p < kHalfKeep; ++p) {
        const int k = 8 * (threadIdx.x + 256 * p);
        if (k < K) put(k, v[p][0], v[p][1]);
    }
    for (int k = 8 * (threadIdx.x + 256 * kHalfKeep); k < K; k += 8 * 256) put(k, *reinterpret_cast<const float4*>(x + k), *reinterpret_cast<const float4*>(x + k + 4));
}

// hidden += the pieces of a projection (nsplit 0: hidden as it lies), and of its RMSNorm the two halves and the rows' largest |x|, as half_split_kernel leaves them; a workgroup a row, which
// stays in registers.  In the place of three launches that each take the row through memory (the sum, the norm, the split): us, 200 rows of 4096 behind eight pieces 6.2 + 8.0 + 5.2,
// 7.2 so.
struct HalfNormArgs { float* hidden; const float* part; int nsplit, H; long long pieces; const float* weight; float eps; _Float16* out; long long plane; float* row_max; };
template <int KEEP>
__global__ __launch_bounds__(1024) void half_norm_split_kernel(const HalfNormArgs a) {
    __shared__ float red[16], top[16];
    float* h = a.hidden + (long long)blockIdx.x * a.H;
    const float* p = a.part + (long long)blockIdx.x * a.H;
    const int bd = (int)blockDim.x;
    float v[KEEP][8];
    float ssq = 0.0f;
    auto get = [](float (&d)[8], const float* src) {
        const float4 x = *reinterpret_cast<const float4*>(src), y = *reinterpret_cast<const float4*>(src + 4);
        d[0] = x.x; d[1] = x.y; d[2] = x.z; d[3] = x.w; d[4] = y.x; d[5] = y.y; d[6] = y.z; d[7] = y.w;
    };
    float w[KEEP][8];
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
        const int k = 8 * ((int)threadIdx.x + bd * u), at = k < a.H ? k : 0;     // (past the row: column 0 again, dropped)
        float old[8];
        get(old, h + at);
        get(w[u], a.weight + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] = 0.0f;
        for (int i = 0; i < a.nsplit; i += 4) {                 // four pieces under way, added in order
            float q[4][8];
#pragma unroll
            for (int c = 0; c < 4; ++c) get(q[c], p + a.pieces * min(i + c, a.nsplit - 1) + at);
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (i + c < a.nsplit)
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[u][e] += q[c][e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[u][e] += old[e];
        if (k < a.H) {
            if (a.nsplit) {
                *reinterpret_cast<float4*>(h + k) = float4{v[u][0], v[u][1], v[u][2], v[u][3]};
                *reinterpret_cast<float4*>(h + k + 4) = float4{v[u][4], v[u][5], v[u][6], v[u][7]};
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) ssq = fmaf(v[u][e], v[u][e], ssq);
        }
    }
    const float inv = 1.0f / sqrtf(block_sum(ssq, red) / (float)a.H + a.eps);
    uint32_t mb = 0;   // (bit patterns: ordered like the values, and a NaN is not dropped)
#pragma unroll
    for (int u = 0; u < KEEP; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[u][e] = v[u][e] * inv * w[u][e];
            if (8 * ((int)threadIdx.x + bd * u) < a.H) mb = max(mb, __float_as_uint(v[u][e]) & 0x7FFFFFFFu);
        }
    const float largest = block_max(__uint_as_float(mb <= 0x7F800000u ? mb : 0x7F800000u), top);
    if (threadIdx.x == 0) a.row_max[blockIdx.x] = largest;
    const float scale = half_scale(largest);
    uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + (long long)blockIdx.x * a.H;
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
        const int k = 8 * ((int)threadIdx.x + bd * u);
        if (k >= a.H) continue;
        uintx4_t b[2];
        TileHalf2::convert(v[u], scale, b);
        *reinterpret_cast<uintx4_t*>(o + k) = b[0];
        *reinterpret_cast<uintx4_t*>(o + a.plane + k) = b[1];
    }
}

// two matrix instructions a product: constants as for bf16 (plan_direct), from 16 .. 200 rows, 1024 .. 28672 outputs, 4096 .. 14336 inputs
static const DirectForm kFormsHalf[] = {{128, 256, 1, 1.65f, 1.65f, 12.0f, 0.6f}, {64, 128, 2, 0.82f, 0.495f, 5.0f, 0.0f}, {64, 64, 2, 0.47f, 0.315f, 4.0f, 0.0f}};
static TilePlan plan_direct_half(int rows, int N, int K, long long room) {
    return plan_direct(kFormsHalf, 3, 64, rows, 1, N, K, room, true);
}
template <int GLU>
static int launch_direct_half(const DirectArgs& d, const TilePlan& p, hipStream_t s, bool sum = true) {
    switch (p.form) {
        case 0: return launch_direct<TileHalf2, 128, 256, 2, 4, 2, GLU, 2>(d, p.splits, s, sum);
        case 1: return launch_direct<TileHalf2, 64, 128, 2, 2, 2, GLU, 2>(d, p.splits, s, sum);
        default: return launch_direct<TileHalf2, 64, 64, 2, 2, 3, GLU, 2>(d, p.splits, s, sum);
    }
}

}  // namespace ntk

using namespace ntk;

static size_t half_row_bytes(int K) { return (size_t)K * 4 + 4; }
// rows of a pass of the direct form: what the workspace and 32-bit offsets hold, in equal passes
static int half_pass_rows(int T, int K, size_t bytes) {
    const long long fit = std::min<long long>({T, ((long long)bytes - 32) / (long long)half_row_bytes(K), ((1LL << 32) - 1) / (K * 2LL), 65535LL});
    const int passes = (T + (int)fit - 1) / (int)fit;
    return (T + passes - 1) / passes;
}
static size_t half_max_bytes(int rows) { return ((size_t)rows * 4 + 15) & ~(size_t)15; }
size_t ntk_gemm_half_many_bytes(int n_tokens, int in_features) { return n_tokens > 0 && in_features > 0 ? (size_t)std::min(n_tokens, 16) * half_row_bytes(in_features) + 32 : 0; }

// a product whose sums are left to its consumer: where they are, or that there are none
static void leave(ntk_gemm_partials* q, float* Y, int rows, int T, int splits, const float* part) {
    *q = ntk_gemm_partials{};
    q->nseg = 1; q->n_tokens = T; q->nsplit = splits; q->part[0] = splits > 1 ? part : nullptr; q->y[0] = Y; q->rows[0] = rows;
}
static int half_many(const ntk_half_desc* d, bool ready, ntk_gemm_partials* defer, void* stream) {
    if (!d || !d->X || d->n < 1 || d->n > 3) return NTK_E_NULL;
    long long N = 0;
    uintptr_t bits = (uintptr_t)d->X | (uintptr_t)d->workspace;
    for (int i = 0; i < d->n; ++i) {
        if (!d->W[i] || (!d->Y[i] && !(d->silu && i))) return NTK_E_NULL;
        if (d->out[i] <= 0) return NTK_E_SHAPE;
        N += d->out[i];
        bits |= (uintptr_t)d->W[i];
    }
    const int T = d->n_tokens, K = d->in_features;
    if (T < 0 || K <= 0 || (d->accumulate && (d->n > 1 || d->silu)) || (d->silu && (d->n != 2 || d->out[0] != d->out[1]))) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    if (!d->workspace) return NTK_E_NULL;
    if (bits & 15) return NTK_E_ALIGN;
    const char *w0 = (const char*)d->W[0], *w1 = (const char*)d->W[1];
    const long long mat = (long long)d->out[0] * K * 2;
    if (K % 64 || K >= 1 << 22 || N > 1 << 30 || (d->silu && std::abs((long long)(w1 - w0)) + mat >= 1LL << 32)) return NTK_E_SHAPE;
    if (d->workspace_bytes < ntk_gemm_half_many_bytes(T, K)) return NTK_E_SHAPE;
    const int per = half_pass_rows(T, K, d->workspace_bytes);
    if ((ready || defer) && per < T) return NTK_E_SHAPE;
    hipStream_t s = resolve_stream(stream);
    for (int t0 = 0; t0 < T; t0 += per) {
        const int n = std::min(per, T - t0);
        const long long plane = (long long)n * K;
        const float* x = d->X + (long long)t0 * K;
        _Float16* halves = (_Float16*)d->workspace;
        char* behind = (char*)d->workspace + 4 * plane;                     // (plane is a multiple of 64)
        float* own_max = (float*)behind;
        behind += half_max_bytes(n);
        if (ready) ;                                                        // (ntk_half_norm_split has left them)
        else if (d->row_max) hipLaunchKernelGGL(half_split_kernel<true>, dim3(n), dim3(256), 0, s, halves, plane, x, K, const_cast<float*>(d->row_max) + t0);
        else hipLaunchKernelGGL(half_split_kernel<false>, dim3(n), dim3(256), 0, s, halves, plane, x, K, own_max);
        DirectArgs a{};
        TileArgs& t = a.t;
        t.W = d->W[0]; t.Y = d->Y[0] + (long long)t0 * d->out[0]; t.ldy = d->out[0]; t.G = 1; t.row_div = 1; t.T = n; t.N = (int)N; t.K = K; t.accumulate = d->accumulate;
        t.row_max = d->row_max && !ready ? d->row_max + t0 : own_max;
        t.part = (float*)behind;
        a.X16 = halves; a.x_row = (uint32_t)K * 2; a.plane = plane * 2;
        const long long left = (char*)d->workspace + d->workspace_bytes - behind;
        const long long room = d->silu || left < 0 ? 0 : left / (long long)sizeof(float);
        const TilePlan p = plan_direct_half(n, (int)N, K, room);
        if (d->silu) {
            t.W = std::min(w0, w1); a.gate_at = (uint32_t)(w0 - (const char*)t.W); a.up_at = (uint32_t)(w1 - (const char*)t.W);
            a.glu_ff = d->out[0];
            launch_direct_half<kGluSilu>(a, p, s);
            continue;
        }
        a.n_seg = d->n;
        for (int i = 0; i < d->n; ++i) { a.segW[i] = d->W[i]; a.segY[i] = d->Y[i] + (long long)t0 * d->out[i]; a.seg_out[i] = d->out[i]; }
        const int splits = launch_direct_half<kGluNone>(a, p, s, !defer);
        if (defer) leave(defer, d->Y[0], (int)N, T, splits, t.part);
    }
    return last_launch_status();
}
int ntk_gemm_half_many(const ntk_half_desc* d, void* stream) { return half_many(d, false, nullptr, stream); }
int ntk_gemm_half_plan(int rows, int N, int K, long long room, int* plan) {
    if (!plan) return NTK_E_NULL;
    if (rows <= 0 || N <= 0 || K <= 0) return NTK_E_SHAPE;
    const TilePlan p = plan_direct_half(rows, N, K, room);
    tell_plan(kFormsHalf[p.form], p, plan);
    return NTK_OK;
}

// ---- a norm's halves from the launch that sums the projection in front of it (include/ntk_engine.h) ----
int ntk_half_norm_takes(int n_tokens, int width, size_t workspace_bytes) {
    return n_tokens > 0 && n_tokens <= 65535 && width > 0 && width % 64 == 0 && width <= 16384 && workspace_bytes >= ntk_gemm_half_many_bytes(n_tokens, width) &&
           half_pass_rows(n_tokens, width, workspace_bytes) == n_tokens;
}
int ntk_half_norm_split(float* hidden, const ntk_gemm_partials* q, const float* weight, int n_tokens, int width, float eps, void* workspace, size_t workspace_bytes, void* stream) {
    if (!hidden || !weight || !workspace) return NTK_E_NULL;
    if (!ntk_half_norm_takes(n_tokens, width, workspace_bytes)) return NTK_E_SHAPE;
    HalfNormArgs a{};
    a.part = hidden;                            // (never read with nsplit 0)
    if (q) {
        if (q->nseg != 1 || q->n_tokens != n_tokens || q->rows[0] != width || q->nsplit < 1) return NTK_E_SHAPE;
        const bool sums = q->nsplit > 1 && q->part[0];
        if (sums || q->y[0] != hidden) { a.part = sums ? q->part[0] : q->y[0]; a.nsplit = sums ? q->nsplit : 1; }
    }
    if (!a.part) return NTK_E_NULL;
    if (((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)a.part) & 15) return NTK_E_ALIGN;
    a.hidden = hidden; a.H = width; a.pieces = (long long)n_tokens * width; a.weight = weight; a.eps = eps;
    a.out = (_Float16*)workspace; a.plane = a.pieces; a.row_max = (float*)((char*)workspace + 4 * a.plane);
    const int threads = width <= 2048 ? 256 : width <= 4096 ? 512 : 1024;
    if (width <= 8 * threads) hipLaunchKernelGGL(half_norm_split_kernel<1>, dim3(n_tokens), dim3(threads), 0, resolve_stream(stream), a);
    else hipLaunchKernelGGL(half_norm_split_kernel<2>, dim3(n_tokens), dim3(threads), 0, resolve_stream(stream), a);
    return last_launch_status();
}
int ntk_gemm_half_normed(const ntk_half_desc* d, ntk_gemm_partials* partials, void* stream) {
    if (d && d->silu && partials) return NTK_E_SHAPE;
    return half_many(d, true, partials, stream);
}

size_t ntk_gemm_half_workspace_bytes(int n_tokens) { return ((size_t)(n_tokens > 0 ? n_tokens : 0) * sizeof(float) + 15) & ~(size_t)15; }

static int gemm_half(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, int accumulate, const float* row_max, void* workspace,
                     size_t workspace_bytes, ntk_gemm_partials* defer, void* stream) {
    if (!Y || !W || !X) return NTK_E_NULL;
    if (n_tokens < 0 || out_features <= 0 || in_features <= 0) return NTK_E_SHAPE;
    if (n_tokens == 0) return NTK_OK;
    const size_t need = !row_max ? ntk_gemm_half_workspace_bytes(n_tokens) : 0;
    if (need && (!workspace || ((uintptr_t)workspace & 15))) return workspace ? NTK_E_ALIGN : NTK_E_NULL;
    if (need > workspace_bytes) return NTK_E_SHAPE;
    hipStream_t s = resolve_stream(stream);
    TileArgs t{};
    t.Y = Y; t.ldy = out_features; t.X = X; t.ldx = in_features; t.W = W; t.row_div = 1; t.G = 1; t.T = n_tokens; t.N = out_features; t.K = in_features; t.accumulate = accumulate;
    t.row_max = row_max;
    long long room = 0;
    if (workspace && !((uintptr_t)workspace & 15) && n_tokens <= 65535) {
        t.part = (float*)((char*)workspace + need);
        room = (long long)((workspace_bytes - need) / sizeof(float));
    }
    const bool vec = in_features % 8 == 0 && in_features < 1 << 24 && !(((uintptr_t)X | (uintptr_t)W) & 15);
    static const TileForm forms[] = {{64, 128, 64, 1.25f, 0.95f}, {32, 64, 64, 0.84f, 0.38f}};
    const TilePlan p = plan_tiles(forms, 2, n_tokens, 1, out_features, in_features, room);
    // The halves formed once, in the workspace, where that is estimated to be ahead: every pass of the rows that it holds reads the weights again, and what the halves take is lost to
    // partial sums.  us over tiles that convert, over halves in a workspace for a third / two thirds / all of the rows / ten times as much: 14336 x 4096, 200 tokens 105, 151 / 89 / 67 / 66;
    // 1024 x 4096, 100 tokens 21 (20 with room for pieces), 145 / 73 / 39 / 18; 4096 x 14336, 200 tokens 207 (112), 426 / 221 / 116 / 69; 2000 tokens 712, 892 / 630 / 463 / 456.  A twentieth in
    // hand for the estimates, a tenth with several passes, a third where the halves leave fewer pieces (1024 x 8192, 2000 tokens: 168 in one piece, 126 in three).  Of 10000 sizes (9 .. 2000
    // rows, 64 .. 28672 outputs) and workspaces with the estimate as it is, those from 1024 inputs on are ahead or within 3 % but for 50, 16 % behind at most (two passes of rows that leave a tile
    // partly empty, 64 outputs); at 256 and 512 inputs, where the launch that forms the halves takes as long as the product, a third of them are behind, by up to 4 us of 12.
    if (vec && workspace && !((uintptr_t)workspace & 15) && in_features % 64 == 0 && in_features < 1 << 22 && workspace_bytes >= ntk_gemm_half_many_bytes(n_tokens, in_features)) {
        const int per = half_pass_rows(n_tokens, in_features, workspace_bytes), passes = (n_tokens + per - 1) / per;
        const long long left = (long long)workspace_bytes - 4LL * per * in_features - (long long)half_max_bytes(per);
        const TilePlan q = plan_direct_half(per, out_features, in_features, std::max(left, 0LL) / (long long)sizeof(float));
        const bool cramped = p.splits > q.splits && left / (long long)sizeof(float) < (long long)p.splits * per * out_features;
        if ((cramped ? 1.35f : passes > 1 ? 1.12f : 1.05f) * passes * (q.us + kSplitUs + (float)per * in_features * 8.0f / kSplitRate) < p.us + kTileUs) {
            ntk_half_desc d{};
            d.W[0] = W; d.Y[0] = Y; d.out[0] = out_features; d.n = 1; d.X = X; d.n_tokens = n_tokens; d.in_features = in_features; d.accumulate = accumulate; d.row_max = row_max;
            d.workspace = workspace; d.workspace_bytes = workspace_bytes;
            return half_many(&d, false, passes == 1 ? defer : nullptr, stream);
        }
    }
    if (need) {
        hipLaunchKernelGGL(token_max_kernel, dim3(n_tokens), dim3(256), 0, s, (float*)workspace, X, in_features);
        t.row_max = (const float*)workspace;
    }
    if (!vec) { launch_tiles<TileHalf2, 64, 64, 2, 2, 2, false>(t, 1, s); return last_launch_status(); }
    const int splits = p.form == 0 ? launch_tiles<TileHalf2, 64, 128, 2, 2, 4, true>(t, p.splits, s, !defer) : launch_tiles<TileHalf2, 32, 64, 2, 2, 2, true>(t, p.splits, s, !defer);
    if (defer) leave(defer, Y, out_features, n_tokens, splits, t.part);
    return last_launch_status();
}
int ntk_gemm_half(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, int accumulate, const float* row_max, void* workspace,
                   size_t workspace_bytes, void* stream) {
    return gemm_half(Y, W, X, n_tokens, out_features, in_features, accumulate, row_max, workspace, workspace_bytes, nullptr, stream);
}
int ntk_gemm_half_defer(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, const float* row_max, void* workspace, size_t workspace_bytes,
                        ntk_gemm_partials* partials, void* stream) {
    if (!partials) return NTK_E_NULL;
    leave(partials, Y, out_features, n_tokens, 1, nullptr);
    return gemm_half(Y, W, X, n_tokens, out_features, in_features, 1, row_max, workspace, workspace_bytes, partials, stream);
}
