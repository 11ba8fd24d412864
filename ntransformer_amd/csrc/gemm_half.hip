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

// two matrix instructions a product: constants as for bf16 (plan_direct), from 16 .. 200 rows, 1024 .. 28672 outputs, 4096 .. 14336 inputs
static TilePlan plan_direct_half(int rows, int N, int K, long long room) {
    static const DirectForm forms[] = {{128, 256, 1, 1.65f, 1.65f, 12.0f}, {64, 128, 2, 0.82f, 0.495f, 5.0f}, {64, 64, 2, 0.47f, 0.315f, 4.0f}};
    return plan_direct(forms, 3, 64, rows, 1, N, K, room);
}
template <int GLU>
static void launch_direct_half(const DirectArgs& d, const TilePlan& p, hipStream_t s) {
    switch (p.form) {
        case 0: launch_direct<TileHalf2, 128, 256, 2, 4, 2, GLU, 2>(d, p.splits, s); break;
        case 1: launch_direct<TileHalf2, 64, 128, 2, 2, 2, GLU, 2>(d, p.splits, s); break;
        default: launch_direct<TileHalf2, 64, 64, 2, 2, 3, GLU, 2>(d, p.splits, s); break;
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

int ntk_gemm_half_many(const ntk_half_desc* d, void* stream) {
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
    hipStream_t s = resolve_stream(stream);
    for (int t0 = 0; t0 < T; t0 += per) {
        const int n = std::min(per, T - t0);
        const long long plane = (long long)n * K;
        const float* x = d->X + (long long)t0 * K;
        _Float16* halves = (_Float16*)d->workspace;
        char* behind = (char*)d->workspace + 4 * plane;                     // (plane is a multiple of 64)
        float* own_max = (float*)behind;
        behind += half_max_bytes(n);
        if (d->row_max) hipLaunchKernelGGL(half_split_kernel<true>, dim3(n), dim3(256), 0, s, halves, plane, x, K, const_cast<float*>(d->row_max) + t0);
        else hipLaunchKernelGGL(half_split_kernel<false>, dim3(n), dim3(256), 0, s, halves, plane, x, K, own_max);
        DirectArgs a{};
        TileArgs& t = a.t;
        t.W = d->W[0]; t.Y = d->Y[0] + (long long)t0 * d->out[0]; t.ldy = d->out[0]; t.G = 1; t.row_div = 1; t.T = n; t.N = (int)N; t.K = K; t.accumulate = d->accumulate;
        t.row_max = d->row_max ? d->row_max + t0 : own_max;
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
        launch_direct_half<kGluNone>(a, p, s);
    }
    return last_launch_status();
}

size_t ntk_gemm_half_workspace_bytes(int n_tokens) { return ((size_t)(n_tokens > 0 ? n_tokens : 0) * sizeof(float) + 15) & ~(size_t)15; }

int ntk_gemm_half(float* Y, const void* W, const float* X, int n_tokens, int out_features, int in_features, int accumulate, const float* row_max, void* workspace,
                   size_t workspace_bytes, void* stream) {
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
    // hand for the estimates, a tenth with several passes, a third where the halves leave fewer pieces (1024 x 8192, 2000 tokens: 168 in one piece, 126 in three).  Over 99 sizes and nine workspaces none is behind the tiles.
    if (vec && workspace && !((uintptr_t)workspace & 15) && in_features % 64 == 0 && in_features < 1 << 22 && workspace_bytes >= ntk_gemm_half_many_bytes(n_tokens, in_features)) {
        const int per = half_pass_rows(n_tokens, in_features, workspace_bytes), passes = (n_tokens + per - 1) / per;
        const long long left = (long long)workspace_bytes - 4LL * per * in_features - (long long)half_max_bytes(per);
        const TilePlan q = plan_direct_half(per, out_features, in_features, std::max(left, 0LL) / (long long)sizeof(float));
        const bool cramped = p.splits > q.splits && left / (long long)sizeof(float) < (long long)p.splits * per * out_features;
        if ((cramped ? 1.35f : passes > 1 ? 1.12f : 1.05f) * passes * (q.us + kSplitUs + (float)per * in_features * 8.0f / kSplitRate) < p.us + kTileUs) {
            ntk_half_desc d{};
            d.W[0] = W; d.Y[0] = Y; d.out[0] = out_features; d.n = 1; d.X = X; d.n_tokens = n_tokens; d.in_features = in_features; d.accumulate = accumulate; d.row_max = row_max;
            d.workspace = workspace; d.workspace_bytes = workspace_bytes;
            return ntk_gemm_half_many(&d, stream);
        }
    }
    if (need) {
        hipLaunchKernelGGL(token_max_kernel, dim3(n_tokens), dim3(256), 0, s, (float*)workspace, X, in_features);
        t.row_max = (const float*)workspace;
    }
    if (!vec) { launch_tiles<TileHalf2, 64, 64, 2, 2, 2, false>(t, 1, s); return last_launch_status(); }
    if (p.form == 0) launch_tiles<TileHalf2, 64, 128, 2, 2, 4, true>(t, p.splits, s);
    else launch_tiles<TileHalf2, 32, 64, 2, 2, 2, true>(t, p.splits, s);
    return last_launch_status();
}
