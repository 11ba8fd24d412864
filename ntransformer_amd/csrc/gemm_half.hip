// gemm_half.hip -- prompt projections over unquantised GGUF weights (F16): Y[t] (+)= W . X[t] for the tokens of a prompt in one pass over W.
// Replaces, for a prompt, the reference's loop of one GEMV per token (attention.cu / ffn.cpp through gemm.cu:32-470): 200 tokens read the weights 200 times, 18 ms a
// layer of an 8B-shaped F16 model against 0.47 ms as tiles (gemm_tile.hip.h); a 200-token pass of eight such layers 144.5 -> 4.1 ms.  Taken from two tokens on: 16 tokens
// through a 4096 x 4096 matrix take 15 us, one token's GEMV 12.  Products on v_mfma_f32_16x16x32_f16; a 32-bit activation goes in as two halves after
// a per-token power of two (largest |x| in [2^14, 2^15)), which is off by at most 2^-23 of the value (a quarter of them by more than 2^-24, where the one-token
// products take all 24 bits), or by 2^-39 of the row's largest where the second half is subnormal.  The sums make up for it (gemm_tile.hip.h): from
// 3072 inputs on a result is as close to 64 bits as the one-token products' (below, those are closer: 2048 inputs 1.22e-7 of the result against 1.10 .. 1.31e-7, 1024 0.98e-7 against 1.04 .. 1.19e-7).
#include "gemm_tile.hip.h"

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

}  // namespace ntk

using namespace ntk;

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
    if (need) {
        hipLaunchKernelGGL(token_max_kernel, dim3(n_tokens), dim3(256), 0, s, (float*)workspace, X, in_features);
        t.row_max = (const float*)workspace;
    }
    if (!vec) { launch_tiles<TileHalf2, 64, 64, 2, 2, 2, false>(t, 1, s); return last_launch_status(); }
    static const TileForm forms[] = {{64, 128, 64, 1.25f, 0.95f}, {32, 64, 64, 0.84f, 0.38f}};
    const TilePlan p = plan_tiles(forms, 2, n_tokens, 1, out_features, in_features, room);
    if (p.form == 0) launch_tiles<TileHalf2, 64, 128, 2, 2, 4, true>(t, p.splits, s);
    else launch_tiles<TileHalf2, 32, 64, 2, 2, 2, true>(t, p.splits, s);
    return last_launch_status();
}
