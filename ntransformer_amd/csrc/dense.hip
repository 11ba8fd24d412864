// dense.hip -- products with dense weight matrices (bfloat16 or float32, row-major [out][in]) for the layer-list model families.
//
// One entry point for a product (ntk_dense) with three kernel forms behind it:
//   * gemm_direct_kernel  more than kGemvRows rows of whole 128-byte chunks (gemm_direct.hip.h), operands from memory straight into LDS: float32 wherever the rows lie in order and
//                         aligned; bf16 where a launch that rounds the activations first and the product over them are estimated faster than tiles (ntk_dense_direct takes rows
//                         that were rounded by whoever wrote them);
//   * gemm_tile_kernel    the other products of more than kGemvRows rows (gemm_tile.hip.h): bf16 weights on v_mfma_f32_16x16x32_bf16, the F32 activations rounded to bfloat16
//                         (nearest even) on their way into LDS; float32 weights on v_mfma_f32_16x16x4_f32 (true 32-bit products and sums); gathered and odd-sized rows;
//   * dense_gemv_kernel   up to kGemvRows rows (decoding): every wave streams a few weight rows at once, 16 bytes per lane and row, the activation
//                         row sits in LDS; bf16 weights are widened exactly and multiplied in F32.  What runs inside the launch on the way in: what the row is still owed (a
//                         sublayer's normed output), an RMS norm; on the way out: a gated unit or an activation.
// Rows can be grouped (a mixture of experts: sorted rows of group g take matrix g) and gathered (row r reads activation row rows[r] / row_div).
// Group sizes live on the device, so the grid covers the worst case and workgroups outside their group's range leave at once.
// A second entry point (ntk_moe_few) runs all of a few tokens' chosen experts, the shared unit and their weighted sum in two row-streaming launches.
#include "gemm_direct.hip.h"
#include "../../include/ntk_layers.h"

namespace ntk {

__device__ __forceinline__ uint16_t f2bf(float f) {   // round to nearest even; NaN stays NaN
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

struct DenseArgs {
    float* Y; int ldy;
    const float* X; int ldx;
    const void* W; long long wstride;
    const int* offsets;
    const int* rows; int row_div;
    int T, N, K, accumulate, G, vec, xvec;   // vec: weight rows 16-byte aligned, K % 8 == 0; xvec: activation rows (and norm_w) 16-byte aligned, K % 4 == 0
    int glu_ff; float glu_limit, glu_alpha, glu_up_offset, glu_cubic;   // few-row form only: outputs f < glu_ff = gated unit of rows f (gate) and glu_ff + f (up)
    const float* norm_w; float norm_eps, norm_offset;   // few-row form only: the activation row is RMS-normed with weight (offset + norm_w) first
    int act;                                            // NTK_ACT_*: on every output
    const float* add_y; int ld_add; const float* add_w; float add_eps, add_mult; float* x_out; int ldxo;   // few-row form only: see ntk_dense_desc
};

constexpr int kActCap = -1;                             // cap * tanh(v / cap), cap in glu_limit: of ntk_dense_capped alone
__device__ __forceinline__ float activate(float v, int act, float cap) {
    if (act == kActCap) return cap * tanhf(v / cap);
    if (act == NTK_ACT_RELU2) { const float p = fmaxf(v, 0.0f); return p * p; }
    return v;
}

// what a product of the few-row forms leaves: s = the wave's sums (lane 63's count), outputs n0 .. of activation row r
template <int RW, bool GLU>
__device__ __forceinline__ void leave_outputs(const DenseArgs& a, const float (&s)[RW], int r, int n0, int n_out) {
    constexpr int OUT = GLU ? RW / 2 : RW;
#pragma unroll
    for (int i = 0; i < OUT; ++i) {
        if (n0 + i >= n_out) continue;
        float t = s[i];
        if constexpr (GLU) {
            const float gg = fminf(s[i], a.glu_limit), uu = fminf(fmaxf(s[i + OUT], -a.glu_limit), a.glu_limit);
            const float zz = a.glu_cubic != 0.0f ? fmaf(a.glu_cubic * gg * gg, gg, gg) : gg;
            t = gg * (1.0f / (1.0f + expf(-a.glu_alpha * zz))) * (uu + a.glu_up_offset);
        }
        float* y = a.Y + (long long)r * a.ldy + n0 + i;
        *y = a.accumulate ? *y + t : activate(t, a.act, a.glu_limit);
    }
}

// ---------------------------------------------------------------------------------------------------------------- few rows: waves stream weight rows
// One workgroup per (group of 4 * RW outputs, activation row): the activation row sits in LDS, each wave owns RW consecutive weight rows and walks
// them together -- per step a lane requests the NEXT 16 bytes of each of its RW rows, then reads its 8 activations once and feeds RW sums from the bytes that
// have arrived; one DPP reduction per row at the end.  The first weights are requested together with the activation row and the weights of its norm, so they
// travel behind the norm's sum over the workgroup.  RW is picked so that the launch still has a few workgroups per CU.
constexpr int kGemvRows = 8;       // up to this many rows take this form
constexpr int kGemvInputs = (160 * 1024 - 1024) / 4;   // ... of up to this many inputs (a row sits in LDS)
template <typename WT, int RW, bool GLU, bool ADD>
__global__ __launch_bounds__(256) void dense_gemv_kernel(const DenseArgs a) {
    extern __shared__ __attribute__((aligned(16))) float xs[];   // the activation row
    const int r = blockIdx.y;
    int g = 0;
    if (a.offsets) {
        if (r >= a.offsets[a.G]) return;
        while (r >= a.offsets[g + 1]) ++g;
    }
    const float* xrow = a.X + (long long)(a.rows ? a.rows[r] / a.row_div : r) * a.ldx;
    const WT* W = (const WT*)a.W + (long long)g * a.wstride;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // GLU: the wave's RW rows are RW / 2 (gate, up) pairs of RW / 2 consecutive outputs
    constexpr int OUT = GLU ? RW / 2 : RW;
    const int n_out = GLU ? a.glu_ff : a.N;
    const int n0 = (blockIdx.x * 4 + wave) * OUT;
    const WT* w[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) {                          // rows past the end re-read the last one and are not stored
        const int row = GLU ? (i < OUT ? min(n0 + i, n_out - 1) : a.glu_ff + min(n0 + i - OUT, n_out - 1)) : min(n0 + i, n_out - 1);
        w[i] = W + (long long)row * a.K;
    }
    constexpr int NV = sizeof(WT) == 2 ? 1 : 2;             // 16-byte pieces of eight weights
    auto weights = [&](uintx4_t (&u)[RW][NV], int k) {
#pragma unroll
        for (int i = 0; i < RW; ++i)
#pragma unroll
            for (int p = 0; p < NV; ++p) u[i][p] = __builtin_nontemporal_load(reinterpret_cast<const uintx4_t*>(w[i] + k) + p);
    };
    __shared__ float red[16];
    float ss = 0.0f;
    uintx4_t first[RW][NV];
    if (a.xvec) {
        // the row's first 4096 entries stay in registers up to the norm; they, their norm weights and the wave's first weights are requested together
        constexpr int XV = 4;
        float4 xv[XV], nv[XV], yv[XV], aw[XV];
        const float* yrow = ADD ? a.add_y + (long long)r * a.ld_add : nullptr;
#pragma unroll
        for (int u = 0; u < XV; ++u) {
            const int k = 4 * (tid + 256 * u);
            if constexpr (ADD) {
                yv[u] = k < a.K ? *reinterpret_cast<const float4*>(yrow + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
                aw[u] = k < a.K ? *reinterpret_cast<const float4*>(a.add_w + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
            }
            xv[u] = k < a.K ? *reinterpret_cast<const float4*>(xrow + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
            nv[u] = a.norm_w && k < a.K ? *reinterpret_cast<const float4*>(a.norm_w + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if (a.vec && lane * 8 < a.K) weights(first, lane * 8);
        for (int k = 4 * (tid + 256 * XV); k < a.K; k += 4 * 256) *reinterpret_cast<float4*>(xs + k) = *reinterpret_cast<const float4*>(xrow + k);
        float inv = 1.0f;
        if constexpr (ADD) {                                // what the row is still owed joins it; the first workgroup of the row leaves the sum
            float sy = 0.0f;
#pragma unroll
            for (int u = 0; u < XV; ++u) { sy = fmaf(yv[u].x, yv[u].x, sy); sy = fmaf(yv[u].y, yv[u].y, sy); sy = fmaf(yv[u].z, yv[u].z, sy); sy = fmaf(yv[u].w, yv[u].w, sy); }
            for (int k = 4 * (tid + 256 * XV); k < a.K; k += 4 * 256)
#pragma unroll
                for (int j = 0; j < 4; ++j) sy = fmaf(yrow[k + j], yrow[k + j], sy);
            const float iy = a.add_mult / sqrtf(block_sum(sy, red) / (float)a.K + a.add_eps);
            float* keep = blockIdx.x == 0 ? a.x_out + (long long)r * a.ldxo : nullptr;
#pragma unroll
            for (int u = 0; u < XV; ++u) {
                const int k = 4 * (tid + 256 * u);
                if (k >= a.K) continue;
                xv[u].x = fmaf(yv[u].x * iy, aw[u].x, xv[u].x); xv[u].y = fmaf(yv[u].y * iy, aw[u].y, xv[u].y);
                xv[u].z = fmaf(yv[u].z * iy, aw[u].z, xv[u].z); xv[u].w = fmaf(yv[u].w * iy, aw[u].w, xv[u].w);
                if (keep) *reinterpret_cast<float4*>(keep + k) = xv[u];
            }
            for (int k = 4 * (tid + 256 * XV); k < a.K; k += 4 * 256)
#pragma unroll
                for (int j = 0; j < 4; ++j) {               // (each thread rewrites what it wrote)
                    xs[k + j] = fmaf(yrow[k + j] * iy, a.add_w[k + j], xs[k + j]);
                    if (keep) keep[k + j] = xs[k + j];
                }
        }
        if (a.norm_w) {                                     // (uniform over the launch)
#pragma unroll
            for (int u = 0; u < XV; ++u) { ss = fmaf(xv[u].x, xv[u].x, ss); ss = fmaf(xv[u].y, xv[u].y, ss); ss = fmaf(xv[u].z, xv[u].z, ss); ss = fmaf(xv[u].w, xv[u].w, ss); }
            for (int k = 4 * (tid + 256 * XV); k < a.K; k += 4 * 256)
#pragma unroll
                for (int j = 0; j < 4; ++j) ss = fmaf(xs[k + j], xs[k + j], ss);
            inv = 1.0f / sqrtf(block_sum(ss, red) / (float)a.K + a.norm_eps);
            for (int k = 4 * (tid + 256 * XV); k < a.K; k += 4 * 256)
#pragma unroll
                for (int j = 0; j < 4; ++j) xs[k + j] = xs[k + j] * inv * (a.norm_offset + a.norm_w[k + j]);   // (each thread rewrites what it wrote)
        }
#pragma unroll
        for (int u = 0; u < XV; ++u) {
            const int k = 4 * (tid + 256 * u);
            if (k >= a.K) continue;
            float4 v = xv[u];
            if (a.norm_w) { v.x = v.x * inv * (a.norm_offset + nv[u].x); v.y = v.y * inv * (a.norm_offset + nv[u].y); v.z = v.z * inv * (a.norm_offset + nv[u].z); v.w = v.w * inv * (a.norm_offset + nv[u].w); }
            *reinterpret_cast<float4*>(xs + k) = v;
        }
    } else {
        if (a.vec && lane * 8 < a.K) weights(first, lane * 8);
        if constexpr (ADD) {
            const float* yrow = a.add_y + (long long)r * a.ld_add;
            float sy = 0.0f;
            for (int k = tid; k < a.K; k += 256) { xs[k] = xrow[k]; sy = fmaf(yrow[k], yrow[k], sy); }
            const float iy = a.add_mult / sqrtf(block_sum(sy, red) / (float)a.K + a.add_eps);
            float* keep = blockIdx.x == 0 ? a.x_out + (long long)r * a.ldxo : nullptr;
            for (int k = tid; k < a.K; k += 256) {
                const float v = fmaf(yrow[k] * iy, a.add_w[k], xs[k]);
                xs[k] = v;
                ss = fmaf(v, v, ss);
                if (keep) keep[k] = v;
            }
        } else {
            for (int k = tid; k < a.K; k += 256) { const float v = xrow[k]; xs[k] = v; ss = fmaf(v, v, ss); }
        }
        if (a.norm_w) {
            ss = block_sum(ss, red);
            const float inv = 1.0f / sqrtf(ss / (float)a.K + a.norm_eps);
            for (int k = tid; k < a.K; k += 256) xs[k] = xs[k] * inv * (a.norm_offset + a.norm_w[k]);   // (each thread rewrites what it wrote)
        }
    }
    __syncthreads();
    if (n0 >= n_out) return;                                // uniform per wave
    float s[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) s[i] = 0.0f;
    if (a.vec) {
        uintx4_t cur[RW][NV], next[RW][NV];
#pragma unroll
        for (int i = 0; i < RW; ++i)
#pragma unroll
            for (int p = 0; p < NV; ++p) cur[i][p] = first[i][p];
        for (int k = lane * 8; k < a.K; k += 64 * 8) {
            if (k + 64 * 8 < a.K) weights(next, k + 64 * 8);        // the next pass's weights behind this pass's sums
            float wv[RW][8];
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                if constexpr (sizeof(WT) == 2) {
                    const uint32_t uu[4] = {cur[i][0].x, cur[i][0].y, cur[i][0].z, cur[i][0].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) { wv[i][2 * j] = __uint_as_float(uu[j] << 16); wv[i][2 * j + 1] = __uint_as_float(uu[j] & 0xffff0000u); }
                } else {
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        wv[i][4 * p] = __uint_as_float(cur[i][p].x); wv[i][4 * p + 1] = __uint_as_float(cur[i][p].y);
                        wv[i][4 * p + 2] = __uint_as_float(cur[i][p].z); wv[i][4 * p + 3] = __uint_as_float(cur[i][p].w);
                    }
                }
            }
            const float4 x0 = *reinterpret_cast<const float4*>(xs + k), x1 = *reinterpret_cast<const float4*>(xs + k + 4);
            const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int i = 0; i < RW; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) s[i] = fmaf(wv[i][j], xv[j], s[i]);
#pragma unroll
            for (int i = 0; i < RW; ++i)
#pragma unroll
                for (int p = 0; p < NV; ++p) cur[i][p] = next[i][p];
        }
    } else {
        for (int k = lane; k < a.K; k += 64) {
            const float xv = xs[k];
#pragma unroll
            for (int i = 0; i < RW; ++i) {
                float wv;
                if constexpr (sizeof(WT) == 2) wv = bf2f(((const uint16_t*)w[i])[k]); else wv = ((const float*)w[i])[k];
                s[i] = fmaf(wv, xv, s[i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) s[i] = wave_sum_lane63(s[i]);
    if (lane == 63) leave_outputs<RW, GLU>(a, s, r, n0, n_out);
}

// ... with the weights read once for R activation rows (a workgroup a row reads them R times, mostly out of the Infinity Cache): the rows' next 1024 columns sit in LDS, a
// lane feeds RW x R sums from a piece of weights.  A row's norm is summed by one wave in the order of the workgroup above, and a sum over k in that kernel's: identical bits.
// Rows on 16 bytes, one group.
constexpr int kRowsStage = 1024;                        // two pieces
template <typename WT, int RW, bool GLU, bool ADD, int R>
__global__ __launch_bounds__(256) void dense_gemv_rows_kernel(const DenseArgs a) {
    extern __shared__ __attribute__((aligned(16))) float xs[];   // [R][columns of a stage]
    __shared__ float scale[2][R];                                // 1 / rms of the rows, and of what they are still owed
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r0 = blockIdx.y * R, live = min(R, a.T - r0);
    constexpr int OUT = GLU ? RW / 2 : RW, NV = sizeof(WT) == 2 ? 1 : 2;
    const int n_out = GLU ? a.glu_ff : a.N, n0 = (blockIdx.x * 4 + wave) * OUT;
    const WT* w[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) {                          // rows past the end re-read the last one and are not stored
        const int row = GLU ? (i < OUT ? min(n0 + i, n_out - 1) : a.glu_ff + min(n0 + i - OUT, n_out - 1)) : min(n0 + i, n_out - 1);
        w[i] = (const WT*)a.W + (long long)row * a.K;
    }
    auto weights = [&](uintx4_t (&u)[RW][NV], int k) {
#pragma unroll
        for (int i = 0; i < RW; ++i)
#pragma unroll
            for (int p = 0; p < NV; ++p) u[i][p] = __builtin_nontemporal_load(reinterpret_cast<const uintx4_t*>(w[i] + k) + p);
    };
    // a ring of pieces of 512 columns of the wave's weights: with the rows in one workgroup there are few waves, and what hides the memory's latency is what each has under way
    constexpr int D = RW >= 4 ? 4 : 8 / RW;
    uintx4_t ring[D][RW][NV];
    auto request = [&](int d, int piece) {
        const int k = piece * 512 + lane * 8;
        if (k < a.K) weights(ring[d], k);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) request(d, d);
    auto x_of = [&](int r) { return a.X + (long long)(a.rows ? a.rows[r] / a.row_div : r) * a.ldx; };
    auto owed = [&](float4 v, int r, int k, float iy) {     // what the row is still owed joins it
        const float4 y = *reinterpret_cast<const float4*>(a.add_y + (long long)r * a.ld_add + k), aw = *reinterpret_cast<const float4*>(a.add_w + k);
        v.x = fmaf(y.x * iy, aw.x, v.x); v.y = fmaf(y.y * iy, aw.y, v.y); v.z = fmaf(y.z * iy, aw.z, v.z); v.w = fmaf(y.w * iy, aw.w, v.w);
        return v;
    };
    // (threads tid, tid + 64, ... of that workgroup are this wave's lanes one after the other; their waves' sums join as block_sum joins them)
    auto sum_of = [&](auto&& at) {
        float part[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float s = 0.0f;
            for (int k = 4 * (lane + 64 * q); k < a.K; k += 1024) {
                const float4 v = at(k);
                s = fmaf(v.x, v.x, s); s = fmaf(v.y, v.y, s); s = fmaf(v.z, v.z, s); s = fmaf(v.w, v.w, s);
            }
            part[q] = wave_sum(s);
        }
        return ((part[0] + part[1]) + part[2]) + part[3];
    };
    if (ADD || a.norm_w)
        for (int j = wave; j < live; j += 4) {
            const int r = r0 + j;
            const float* x = x_of(r);
            float iy = 0.0f, inv = 1.0f;
            if constexpr (ADD) iy = a.add_mult / sqrtf(sum_of([&](int k) { return *reinterpret_cast<const float4*>(a.add_y + (long long)r * a.ld_add + k); }) / (float)a.K + a.add_eps);
            if (a.norm_w)
                inv = 1.0f / sqrtf(sum_of([&](int k) {
                          const float4 v = *reinterpret_cast<const float4*>(x + k);
                          return ADD ? owed(v, r, k, iy) : v;
                      }) / (float)a.K + a.norm_eps);
            if (lane == 0) { scale[0][j] = inv; scale[1][j] = iy; }
        }
    float s[R][RW] = {};
    float4 ahead[R];                                        // the next stage's columns of the rows, four a thread
    auto fetch = [&](int k0) {
        const int k = k0 + 4 * tid;
        if (k < a.K)
#pragma unroll
            for (int j = 0; j < R; ++j) ahead[j] = *reinterpret_cast<const float4*>(x_of(r0 + min(j, live - 1)) + k);
    };
    auto stage = [&](int k0) {                              // `ahead` into LDS, finished; the stage behind it requested
        __syncthreads();
        const int k = k0 + 4 * tid;
        if (k < a.K) {
            const float4 nw = a.norm_w ? *reinterpret_cast<const float4*>(a.norm_w + k) : float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < R; ++j) {
                const int r = r0 + min(j, live - 1);
                float4 v = ahead[j];
                if constexpr (ADD) {
                    v = owed(v, r, k, scale[1][min(j, live - 1)]);
                    if (blockIdx.x == 0 && j < live) *reinterpret_cast<float4*>(a.x_out + (long long)r * a.ldxo + k) = v;
                }
                if (a.norm_w) {
                    const float inv = scale[0][min(j, live - 1)];
                    v.x = v.x * inv * (a.norm_offset + nw.x); v.y = v.y * inv * (a.norm_offset + nw.y); v.z = v.z * inv * (a.norm_offset + nw.z); v.w = v.w * inv * (a.norm_offset + nw.w);
                }
                *reinterpret_cast<float4*>(xs + j * kRowsStage + 4 * tid) = v;
            }
        }
        __syncthreads();
        fetch(k0 + kRowsStage);
    };
    fetch(0);
    __syncthreads();
    const int pieces = (a.K + 511) / 512;
    for (int p0 = 0; p0 < pieces; p0 += D)
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int p = p0 + d, k = p * 512 + lane * 8;
            if (p >= pieces) break;                         // (uniform)
            if (d % 2 == 0) stage(p * 512);
            if (k < a.K) {
                float wv[RW][8];
#pragma unroll
                for (int i = 0; i < RW; ++i) {
                    if constexpr (sizeof(WT) == 2) {
                        const uint32_t uu[4] = {ring[d][i][0].x, ring[d][i][0].y, ring[d][i][0].z, ring[d][i][0].w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) { wv[i][2 * e] = __uint_as_float(uu[e] << 16); wv[i][2 * e + 1] = __uint_as_float(uu[e] & 0xffff0000u); }
                    } else {
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            wv[i][4 * q] = __uint_as_float(ring[d][i][q].x); wv[i][4 * q + 1] = __uint_as_float(ring[d][i][q].y);
                            wv[i][4 * q + 2] = __uint_as_float(ring[d][i][q].z); wv[i][4 * q + 3] = __uint_as_float(ring[d][i][q].w);
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    const float* xj = xs + j * kRowsStage + (d & 1) * 512 + lane * 8;
                    const float4 x0 = *reinterpret_cast<const float4*>(xj), x1 = *reinterpret_cast<const float4*>(xj + 4);
                    const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
                    for (int i = 0; i < RW; ++i)
#pragma unroll
                        for (int e = 0; e < 8; ++e) s[j][i] = fmaf(wv[i][e], xv[e], s[j][i]);
                }
            }
            request(d, p + D);
        }
    if (n0 >= n_out) return;
#pragma unroll
    for (int j = 0; j < R; ++j) {
#pragma unroll
        for (int i = 0; i < RW; ++i) s[j][i] = wave_sum_lane63(s[j][i]);
        if (lane == 63 && j < live) leave_outputs<RW, GLU>(a, s[j], r0 + j, n0, n_out);
    }
}

// ---------------------------------------------------------------------------------------------------------------- a few tokens' experts
// Two launches for everything between a router and the sum of its experts (see ntk_moe_few).  The first streams weight rows like dense_gemv_kernel: a wave
// owns RW rows (pairs of rows), the next pass's 16 bytes per lane and row are requested before the current ones are used, the first ones ahead of the row's way into LDS.
struct MoeFewArgs {
    float* out; int ldo;
    const float* h; int ldh;
    const int* ids; const float* wts; int top, experts;
    const void *up, *down, *shared_up, *shared_down; int ff, shared_ff;
    const float* sgate;
    int act; float* mid; int n, vec;
    float limit, shared_limit, alpha, up_offset;    // GLU: see ntk_moe_few_desc
    const float* mix; int ld_mix;
};

template <typename WT> struct WeightPiece {                  // eight weights of a row
    static constexpr int NV = sizeof(WT) == 2 ? 1 : 2;
    uintx4_t u[NV];
    __device__ __forceinline__ void load(const WT* p) {
#pragma unroll
        for (int i = 0; i < NV; ++i) u[i] = __builtin_nontemporal_load(reinterpret_cast<const uintx4_t*>(p) + i);
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < NV; ++i) u[i] = uintx4_t{0u, 0u, 0u, 0u};
    }
    __device__ __forceinline__ float dot(const float* x, float s) const {      // s + the eight products, k ascending; x 16-byte aligned
        const float4 x0 = *reinterpret_cast<const float4*>(x), x1 = *reinterpret_cast<const float4*>(x + 4);
        const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
        if constexpr (sizeof(WT) == 2) {
            const uint32_t w[4] = {u[0].x, u[0].y, u[0].z, u[0].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) { s = fmaf(__uint_as_float(w[j] << 16), xv[2 * j], s); s = fmaf(__uint_as_float(w[j] & 0xffff0000u), xv[2 * j + 1], s); }
        } else {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                s = fmaf(__uint_as_float(u[p].x), xv[4 * p], s); s = fmaf(__uint_as_float(u[p].y), xv[4 * p + 1], s);
                s = fmaf(__uint_as_float(u[p].z), xv[4 * p + 2], s); s = fmaf(__uint_as_float(u[p].w), xv[4 * p + 3], s);
            }
        }
        return s;
    }
};
template <typename WT> __device__ __forceinline__ float weight_value(const WT* p) {
    if constexpr (sizeof(WT) == 2) return bf2f(*p); else return *p;
}

// mid[t][slot * ff + f] = act(U_e h)[f] times the expert's weight for the token's chosen experts, then the shared unit's times its gate; grid (rows / (4 RW), T).
// GLU: a unit's matrix holds its gate rows, then its up rows; a wave walks RW pairs of them.
template <typename WT, int RW, bool GLU>
__global__ __launch_bounds__(256) void moe_few_up_kernel(const MoeFewArgs a) {
    extern __shared__ __attribute__((aligned(16))) float xs[];   // the token's row
    constexpr int NR = GLU ? 2 * RW : RW;                     // weight rows of a wave
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int routed = a.top * a.ff, rows = routed + a.shared_ff, m0 = (blockIdx.x * 4 + wave) * RW;
    const int* ids = a.ids + (long long)t * a.top;
    const WT* w[NR];
    bool any = false;
#pragma unroll
    for (int i = 0; i < RW; ++i) {                            // rows of identity experts and rows past the end: nothing to read
        const int m = m0 + i;
        w[i] = nullptr;
        int ff = 0;
        if (m < routed) {
            const int e = ids[m / a.ff];
            ff = a.ff;
            if (e >= 0 && e < a.experts) w[i] = (const WT*)a.up + ((long long)e * (GLU ? 2 : 1) * a.ff + m % a.ff) * a.n;
        } else if (m < rows) {
            ff = a.shared_ff;
            w[i] = (const WT*)a.shared_up + (long long)(m - routed) * a.n;
        }
        if constexpr (GLU) w[RW + i] = w[i] ? w[i] + (long long)ff * a.n : nullptr;
        any = any || w[i];
    }
    WeightPiece<WT> cur[NR], next[NR];
    auto request = [&](WeightPiece<WT>(&p)[NR], int k) {
#pragma unroll
        for (int i = 0; i < NR; ++i) { if (w[i]) p[i].load(w[i] + k); else p[i].clear(); }
    };
    if (a.vec && lane * 8 < a.n) request(cur, lane * 8);
    const float* x = a.h + (long long)t * a.ldh;
    if (a.vec)
        for (int k = 4 * tid; k < a.n; k += 4 * 256) *reinterpret_cast<float4*>(xs + k) = *reinterpret_cast<const float4*>(x + k);
    else
        for (int k = tid; k < a.n; k += 256) xs[k] = x[k];
    __syncthreads();
    if (!any) return;                                         // (uniform over the wave)
    float s[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) s[i] = 0.0f;
    if (a.vec) {
        for (int k = lane * 8; k < a.n; k += 512) {
            if (k + 512 < a.n) request(next, k + 512);
#pragma unroll
            for (int i = 0; i < NR; ++i) { s[i] = cur[i].dot(xs + k, s[i]); cur[i] = next[i]; }
        }
    } else {
        for (int k = lane; k < a.n; k += 64)
#pragma unroll
            for (int i = 0; i < NR; ++i)
                if (w[i]) s[i] = fmaf(weight_value(w[i] + k), xs[k], s[i]);
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) s[i] = wave_sum_lane63(s[i]);
#pragma unroll
    for (int i = 0; i < RW; ++i) {
        if (lane == 63 && w[i]) {
            const bool chosen = m0 + i < routed;
            const float wt = chosen ? a.wts[(long long)t * a.top + (m0 + i) / a.ff] : a.sgate ? a.sgate[t] : 1.0f;
            float v;
            if constexpr (GLU) {
                const float limit = chosen ? a.limit : a.shared_limit, g = fminf(s[i], limit), u = fminf(fmaxf(s[RW + i], -limit), limit);
                v = g * (1.0f / (1.0f + expf(-a.alpha * g))) * (u + a.up_offset);
            } else v = activate(s[i], a.act, 0.0f);
            a.mid[(long long)t * rows + m0 + i] = v * wt;
        }
    }
}

// out[t][i] = one row of weights [D_e0[i] | D_e1[i] | ... | Ds[i]] against the weighted activations side by side; grid (n / kDownRows, T).  Bound by the weights'
// stream.  A row is a list of passes of 512 entries inside one segment (a chosen expert, the shared unit; identity experts are passed over); the workgroup's four
// waves take every fourth pass of the same kDownRows rows, so the activations go straight from the caches into registers, once for the rows -- staging all of
// them in LDS, as it was, put a 45 KB copy per workgroup before the first product -- and the requests of DEPTH passes are under way.  2048 outputs of six bf16
// experts of 1408 and a shared unit of 2816 (46 MB): 20.5 us -> 10.5 us, 4.4 TB/s.
constexpr int kDownRows = 4;
template <typename WT, int DEPTH>
__global__ __launch_bounds__(256) void moe_few_down_kernel(const MoeFewArgs a) {
    constexpr int RW = kDownRows;
    __shared__ float part[4][RW];
    const int t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int routed = a.top * a.ff, K = routed + a.shared_ff, i0 = blockIdx.x * RW;
    const int* ids = a.ids + (long long)t * a.top;
    const float* mid = a.mid + (long long)t * K;
    // the pass that is requested next: segment (`top` = the shared unit, top + 1 = past the end), its matrix, the pass's first entry in it -- uniform over the wave
    int seg = -1, k0 = 0, len = 0;
    const WT* mat = nullptr;
    auto next_segment = [&]() {
        for (++seg; seg < a.top; ++seg) {
            const int e = ids[seg];
            if (e >= 0 && e < a.experts) { mat = (const WT*)a.down + (long long)e * a.n * a.ff; len = a.ff; return; }
        }
        if (seg == a.top && a.shared_ff > 0) { mat = (const WT*)a.shared_down; len = a.shared_ff; return; }
        seg = a.top + 1;
    };
    auto settle = [&]() {                                     // k0 counts on past a segment's last pass into the next one's
        while (seg <= a.top && k0 >= len) { k0 -= (len + 511) & ~511; next_segment(); }
    };
    float s[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) s[i] = 0.0f;
    next_segment();
    if (a.vec) {
        WeightPiece<WT> piece[DEPTH][RW];
        float4 x[DEPTH][2];
        bool have[DEPTH];
        auto request = [&](int d) {
            have[d] = seg <= a.top;
            if (!have[d]) return;
            const int k = k0 + lane * 8;
            if (k < len) {
                const float* xp = mid + (seg < a.top ? seg * a.ff : routed) + k;
                x[d][0] = *reinterpret_cast<const float4*>(xp);
                x[d][1] = *reinterpret_cast<const float4*>(xp + 4);
#pragma unroll
                for (int i = 0; i < RW; ++i) piece[d][i].load(mat + (long long)min(i0 + i, a.n - 1) * len + k);   // (rows past the end re-read the last one and are not stored)
            } else {
                x[d][0] = x[d][1] = float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < RW; ++i) piece[d][i].clear();
            }
            k0 += 4 * 512;
            settle();
        };
        k0 = wave * 512;
        settle();
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) request(d);
        while (have[0]) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                if (have[d]) {
                    const float xv[8] = {x[d][0].x, x[d][0].y, x[d][0].z, x[d][0].w, x[d][1].x, x[d][1].y, x[d][1].z, x[d][1].w};
#pragma unroll
                    for (int i = 0; i < RW; ++i) s[i] = piece[d][i].dot(xv, s[i]);
                    request(d);
                }
            }
        }
    } else {
        if (a.ff >= 512) {
            for (; seg <= a.top; next_segment())
                for (int k = tid; k < len; k += 256)
#pragma unroll
                    for (int i = 0; i < RW; ++i) s[i] = fmaf(weight_value(mat + (long long)min(i0 + i, a.n - 1) * len + k), mid[(seg < a.top ? seg * a.ff : routed) + k], s[i]);
        } else
        // (short segments: entries of all as one row, four under way -- segment by segment each one's first entries are waited for: 6 choices of 33, width 300: 10.0 us / 7.7; of 1403, width 1001,
        // 28 / 36)
        for (int e0 = tid; e0 < K; e0 += 4 * 256) {
            float x[4], w[4][RW];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + 256 * u, sl = e < routed ? e / a.ff : a.top, id = e < routed ? ids[sl] : 0;
                const bool in = e < K && (sl == a.top || (id >= 0 && id < a.experts));
                x[u] = 0.0f;
#pragma unroll
                for (int i = 0; i < RW; ++i) w[u][i] = 0.0f;
                if (in) {
                    const int k = sl < a.top ? e - sl * a.ff : e - routed, width = sl < a.top ? a.ff : a.shared_ff;
                    const WT* m = sl < a.top ? (const WT*)a.down + (long long)id * a.n * a.ff : (const WT*)a.shared_down;
                    x[u] = mid[e];
#pragma unroll
                    for (int i = 0; i < RW; ++i) w[u][i] = weight_value(m + (long long)min(i0 + i, a.n - 1) * width + k);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < RW; ++i) s[i] = fmaf(w[u][i], x[u], s[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
        s[i] = wave_sum_lane63(s[i]);
        if (lane == 63) part[wave][i] = s[i];
    }
    __syncthreads();
    if (tid >= RW || i0 + tid >= a.n) return;
    float ident = 0.0f;                                       // the weights of the token's identity experts
    for (int sl = 0; sl < a.top; ++sl)
        if (ids[sl] >= a.experts) ident += a.wts[(long long)t * a.top + sl];
    float v = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
    if (ident != 0.0f) v = fmaf(ident, a.h[(long long)t * a.ldh + i0 + tid], v);
    float* o = a.out + (long long)t * a.ldo + i0 + tid;
    if (a.mix) v += a.mix[(long long)t * a.ld_mix + i0 + tid] + *o;
    *o = v;
}

template <typename WT>
static void launch_moe_few(const MoeFewArgs& a, int T, bool glu, hipStream_t s) {
    const int rows = a.top * a.ff + a.shared_ff;
    const size_t lu = ((size_t)a.n * 4 + 15) & ~(size_t)15;
    if (glu) hipLaunchKernelGGL((moe_few_up_kernel<WT, 2, true>), dim3((rows + 7) / 8, T), dim3(256), lu, s, a);
    else hipLaunchKernelGGL((moe_few_up_kernel<WT, 2, false>), dim3((rows + 7) / 8, T), dim3(256), lu, s, a);
    hipLaunchKernelGGL((moe_few_down_kernel<WT, 3>), dim3((a.n + kDownRows - 1) / kDownRows, T), dim3(256), 0, s, a);
}

// Which launches of 2 .. 8 rows read their weights once.  The other form's rows run side by side while a few workgroups a CU hold them all (2048 outputs of bf16 up to five rows), and a norm is
// formed there by a workgroup, here by a wave; what is saved are the weights' further passes, of which bf16 has half.  us, a workgroup a row / this, rows 2, 4, 8: bf16 2048 x 2048 5.3 / 4.6,
// 5.5 / 5.6, 9.0 / 7.7; 6144 x 2048 8.0 / 7.4, 14.6 / 9.2, 25 / 12; behind a norm 9.2 / 9.0, 15.7 / 10.9, 28 / 15; 2048 x 2048 behind one 5.8 / 6.3, 6.4 / 7.6, 10.3 / 11.0; float32 2048 x 2048 8.1 / 6.2,
// 13.2 / 7.3, 23 / 9.6, behind a norm and a sum 9.8 / 10.2, 14.1 / 12.0, 24 / 18; gated units with both, bf16 1408 x 2048 7.5 / 9.7, 8.8 / 11.7, 12 / 19, 7488 x 2048 27 / 24, 44 / 29, 81 / 46;
// float32 10.8 / 12.5, 18 / 15, 31 / 22 and 48 / 36, 91 / 42, 171 / 57.  With few outputs the other form's rows fill CUs that this one leaves idle, and a norm's waves walk all its inputs: float32, 8
// rows, 256 x 4096 6.5 / 10.8, 512 x 8192 17 / 20, behind a norm 256 x 14336 21 / 52, 704 x 4096 14 / 17, and 1024 x 4096, 2 rows, 8.6 / 10.0; with a sum 1024 x 4096, 4 rows, 13 / 17; units of
// 704 x 4096, 4 rows, 18 / 20.  bf16 units, rows 2, 5, 8: 4096 x 3072 16 / 18, 34 / 27, 53 / 32; 4608 x 2560 17 / 18, 33 / 42, 52 / 50; 6144 x 2560 20 / 19, 46 / 43, 70 / 51.
// Of 5194 launches of 512 .. 14336 inputs, 1024 .. 32000 outputs and 2 .. 8 rows that this takes four are behind the other form by more than 2 %, by 5 % at most.
template <typename WT, bool ADD>
static bool rows_share_weights(const DenseArgs& a, int rows) {
    if (rows < 2 || !a.vec || !a.xvec || a.offsets) return false;
    const long long n = a.glu_ff > 0 ? a.glu_ff : a.N, size = n * a.K;
    if constexpr (sizeof(WT) == 2) {
        const bool normed = ADD || a.norm_w;
        if (a.glu_ff == 0) return size >= 4LL << 20 && n * rows >= (size >= 8LL << 20 && !normed ? 12288 : 16384) && (n >= 4096 || !normed);
        if (rows == 2) return n >= 6144 && a.K >= 2048;
        const long long groups = (n + 15) / 16;      // (from five rows on one a CU at a time: two rounds are worth it from three quarters of their places on)
        if (rows > 4 && rows < 8 && (size < 10000000 || 4 * groups < 3 * ((groups + 255) / 256 * 256))) return false;
        return n >= 4096 && size >= 8LL << 20;
    }
    if (a.glu_ff > 0) return size >= 2800000 && n >= 1024 && (rows >= 3 || n >= 4096);
    if constexpr (ADD) return size >= 4LL << 20 && n >= 2048 && (rows >= 4 || n >= 4096);
    if (a.norm_w) return size >= 2LL << 20 && (n >= 2048 || (n >= 1024 && n * rows >= 8192));
    return size >= 1LL << 20 && n >= 1024;
}

template <typename WT, bool ADD>
static void launch_gemv(const DenseArgs& a, int rows, hipStream_t s) {
    const size_t lds = ((size_t)a.K * 4 + 15) & ~(size_t)15;
    // Rows per wave, measured over layer-like shapes (2048 .. 64000 outputs of 768 .. 4096 inputs, 1 .. 6 activation rows): two rows per wave are
    // the best or within noise everywhere from 4096 outputs x rows on (a 64000 x 4096 head: 84 us against 98 with one or eight), one below; launches
    // under ~20 MB sit at 4 - 6 us whatever the choice.  The GLU form keeps pairs: 4 pairs per wave for the large expert launches.
    if (rows_share_weights<WT, ADD>(a, rows)) {
        auto go = [&](auto rw, auto glu, auto r) {
            constexpr int RW = decltype(rw)::value, R = decltype(r)::value;
            constexpr bool GLU = decltype(glu)::value;
            const int n = GLU ? a.glu_ff : a.N, out = 4 * (GLU ? RW / 2 : RW);
            hipLaunchKernelGGL((dense_gemv_rows_kernel<WT, RW, GLU, ADD, R>), dim3((n + out - 1) / out, (rows + R - 1) / R), dim3(256), (size_t)R * kRowsStage * 4, s, a);
        };
        using Yes = std::true_type; using No = std::false_type;
        using C1 = std::integral_constant<int, 1>; using C2 = std::integral_constant<int, 2>; using C4 = std::integral_constant<int, 4>;
        auto pick = [&](auto r) {
            if (a.glu_ff >= 4096) go(C4{}, Yes{}, r);
            else if (a.glu_ff > 0) go(C2{}, Yes{}, r);
            else if (a.N >= 4096) go(C2{}, No{}, r);
            else go(C1{}, No{}, r);
        };
        if (rows == 2) pick(C2{});
        else if (rows == 3) pick(std::integral_constant<int, 3>{});
        else if (rows == 4) pick(C4{});
        else if (rows <= 6) pick(std::integral_constant<int, 6>{});
        else pick(std::integral_constant<int, 8>{});
        return;
    }
    const long long work = (long long)a.N * rows;
    int rw = work >= 4096 ? 2 : 1;
    if (const int force = NTK_TUNE_ENV_INT("NTK_DENSE_GEMV_RW", 0)) rw = force;   // (tuning builds only)
    if (a.glu_ff > 0) {
        const int out = work >= 4 * 8 * 512 ? 4 : work >= 4 * 4 * 512 ? 2 : 1;   // (gate, up) pairs per wave
        const dim3 grid((a.glu_ff + 4 * out - 1) / (4 * out), rows, 1);
        if (out == 4) hipLaunchKernelGGL((dense_gemv_kernel<WT, 8, true, ADD>), grid, dim3(256), lds, s, a);
        else if (out == 2) hipLaunchKernelGGL((dense_gemv_kernel<WT, 4, true, ADD>), grid, dim3(256), lds, s, a);
        else hipLaunchKernelGGL((dense_gemv_kernel<WT, 2, true, ADD>), grid, dim3(256), lds, s, a);
        return;
    }
    const dim3 grid((a.N + 4 * rw - 1) / (4 * rw), rows, 1);
    if (rw == 8) hipLaunchKernelGGL((dense_gemv_kernel<WT, 8, false, ADD>), grid, dim3(256), lds, s, a);
    else if (rw == 4) hipLaunchKernelGGL((dense_gemv_kernel<WT, 4, false, ADD>), grid, dim3(256), lds, s, a);
    else if (rw == 2) hipLaunchKernelGGL((dense_gemv_kernel<WT, 2, false, ADD>), grid, dim3(256), lds, s, a);
    else hipLaunchKernelGGL((dense_gemv_kernel<WT, 1, false, ADD>), grid, dim3(256), lds, s, a);
}

// x rounded to bfloat16, eight values a thread (V: 16-byte pieces of both; else one by one)
template <bool V>
__global__ __launch_bounds__(256) void round_rows_kernel(uint16_t* y, int ldy, const float* x, int ldx, int pieces, int n, long long total) {
    const long long i = blockIdx.x * 256LL + threadIdx.x;
    if (i >= total) return;
    const long long t = i / pieces;
    const int k = (int)(i - t * pieces) * 8;
    const float* xr = x + t * ldx + k;
    uint16_t* yr = y + t * ldy + k;
    if constexpr (V) {
        const float4 u = *reinterpret_cast<const float4*>(xr), v = *reinterpret_cast<const float4*>(xr + 4);
        *reinterpret_cast<uintx4_t*>(yr) = uintx4_t{pack_bf16(u.x, u.y), pack_bf16(u.z, u.w), pack_bf16(v.x, v.y), pack_bf16(v.z, v.w)};
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) if (k + j < n) yr[j] = (uint16_t)pack_bf16(xr[j], 0.0f);
    }
}

// ---- bf16 products over operands in memory (gemm_direct.hip.h)
constexpr float kRoundUs = 3.5f, kRoundRate = 4e6f;     // the launch that rounds a product's activations: us, and bytes per us (six an entry)
static const DirectForm kFormsBf16[] = {{256, 256, 1, 1.45f, 1.45f, 12.0f}, {256, 128, 1, 0.84f, 0.84f, 9.0f}, {128, 256, 1, 0.85f, 0.85f, 9.0f}, {128, 128, 2, 0.72f, 0.475f, 7.0f},
                                        {128, 128, 1, 0.50f, 0.57f, 7.0f}, {64, 128, 2, 0.42f, 0.35f, 5.0f}, {64, 64, 3, 0.33f, 0.22f, 4.0f}};
static TilePlan plan_direct_bf16(int rows, int groups, int N, int K, long long room) {
    return plan_direct(kFormsBf16, 7, 64, rows, groups, N, K, room, groups == 1);
}
// float32: K in chunks of 32; one form, ahead of larger and smaller tiles and other splits of the tile over waves at the sizes they were tried at (12 .. 200 rows, 900 in 32 groups).  Over 337
// grouped sizes it takes 0.89 of gemm_tile.hip.h's time on average and is 3 .. 17 % behind it at about eleven (40 rows in 128 groups, 300 in 8 or 16).  us, the form of gemm_tile.hip.h
// before -> now: 150 x 14976 x 2048 114 -> 91 (101 TF/s of the 153 a large library product reaches), 150 x 2048 x 7488 58 -> 49, 150 x 6240 x 2048 51 -> 39, 12 x 2048 x 2048 11 -> 9
static TilePlan plan_direct_f32(int rows, int groups, int N, int K, long long room) {
    static const DirectForm form[] = {{32, 64, 4, 0.38f, 0.27f, 4.0f}};
    return plan_direct(form, 1, 32, rows, groups, N, K, room);
}
template <int GLU>
static void launch_direct_f32(const DirectArgs& d, int groups, long long room, hipStream_t s) {
    launch_direct<TileF32, 32, 64, 2, 2, 3, GLU, 4>(d, plan_direct_f32(d.t.T, groups, d.t.N, d.t.K, room).splits, s);
}
static TilePlan plan_tiles_bf16(int rows, int groups, int N, int K, long long room) {
    static const TileForm forms[] = {{128, 128, 32, 0.65f, 0.43f}, {64, 128, 64, 0.80f, 0.68f}, {64, 64, 64, 0.70f, 0.35f}, {32, 64, 64, 0.60f, 0.22f}};
    return plan_tiles(forms, 4, rows, groups, N, K, room);
}
template <int GLU>
static void launch_direct_bf16(const DirectArgs& d, const TilePlan& p, hipStream_t s) {
    switch (p.form) {
        case 0: launch_direct<TileBf16, 256, 256, 4, 2, 2, GLU, 2>(d, p.splits, s); break;
        case 1: launch_direct<TileBf16, 256, 128, 4, 2, 3, GLU, 2>(d, p.splits, s); break;
        case 2: launch_direct<TileBf16, 128, 256, 2, 4, 3, GLU, 2>(d, p.splits, s); break;
        case 3: launch_direct<TileBf16, 128, 128, 4, 2, 2, GLU, 4>(d, p.splits, s); break;
        case 4: launch_direct<TileBf16, 128, 128, 4, 2, 4, GLU, 2>(d, p.splits, s); break;
        case 5: launch_direct<TileBf16, 64, 128, 2, 2, 3, GLU, 2>(d, p.splits, s); break;
        default: launch_direct<TileBf16, 64, 64, 2, 2, 3, GLU, 3>(d, p.splits, s); break;
    }
}

}  // namespace ntk

using namespace ntk;

int ntk_round_rows(void* y, int ldy, const float* x, int ldx, int T, int n, void* stream) {
    if (!y || !x) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const int pieces = (n + 7) / 8;
    const long long total = (long long)T * pieces;
    const bool vec = n % 8 == 0 && ldy % 8 == 0 && ldx % 4 == 0 && !(((uintptr_t)y | (uintptr_t)x) & 15);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (vec) hipLaunchKernelGGL(round_rows_kernel<true>, grid, dim3(256), 0, resolve_stream(stream), (uint16_t*)y, ldy, x, ldx, pieces, n, total);
    else hipLaunchKernelGGL(round_rows_kernel<false>, grid, dim3(256), 0, resolve_stream(stream), (uint16_t*)y, ldy, x, ldx, pieces, n, total);
    return last_launch_status();
}

// whole chunks of 128 bytes, rows that 32-bit offsets reach, and a one-dimensional grid of tiles that fits: 2^32 threads, 256 for 32 x 64 results, with room for the groups' tiles
int ntk_dense_direct_takes(int wdtype, int T, int x16_rows, int N, int K) {
    const int es = wdtype == NTK_DT_BF16 ? 2 : 4;
    return (wdtype == NTK_DT_BF16 || wdtype == NTK_DT_F32) && T > kGemvRows && N > 0 && K > 0 && K % (128 / es) == 0 && (long long)N * K * es < 1LL << 32 && (long long)x16_rows * K * es < 1LL << 32 &&
           (T / 32 + 1LL) * (N / 64 + 1LL) < 1LL << 23;
}

// A unit's first product leaves its activations in its epilogue in the direct form, so its inputs are not cut into pieces: with few tiles and long rows that costs more than the launch
// that it saves.  us of a unit through ntk_dense, ntk_glu and ntk_dense / directly, 33 rows: 4096 inputs, 512 values bf16 17.7 / 28.4, float32 25.2 / 63.5; 2048, 2816 24.7 / 23.3, 41.4 /
// 43.3; 2048, 7488 35.7 / 27.1, 84.0 / 64.8.  In groups neither form cuts, and what is left to lose are units of a few values and, without a gate, the launch that the rounding adds.  Over
// 3076 bf16 units (192 .. 4096 inputs, 128 .. 7488 values, 9 .. 1000 tokens, 1 .. 64 groups) always direct was behind by more than 3 % in 668, by up to 2.4 times, with 0.87 of the time
// on average; so in 12, by 11 % at most, with 0.86.  Over 270 float32 units of one matrix 113 and up to 3.6 times, 1.09; so none, 0.85.
int ntk_dense_unit_direct(int wdtype, int rows, int groups, int tokens, int width, int ff, int plain, size_t scratch_bytes) {
    if (rows <= kGemvRows || groups <= 0 || tokens <= 0 || width <= 0 || ff <= 0) return 0;
    const int first = plain ? ff : 2 * ff;
    const long long room = groups > 1 || rows > 65535 ? 0 : (long long)(scratch_bytes / sizeof(float));
    const float glu = plain ? 0.0f : 3.5f + (float)rows * ff * 12.0f / 4e6f;
    if (wdtype == NTK_DT_F32)
        return !plain && (groups > 1 || plan_direct_f32(rows, 1, first, width, 0).us <= plan_direct_f32(rows, 1, first, width, room).us + glu - 2.5f);
    if (groups > 1 && ff < (plain ? 640 : 256)) return 0;
    if (groups > 1 && !plain) return 1;
    const float direct = plan_direct_bf16(rows, groups, first, width, 0).us + plan_direct_bf16(rows, groups, width, ff, room).us + kRoundUs + (float)tokens * width * 6.0f / kRoundRate;
    const float tiles = plan_tiles_bf16(rows, groups, first, width, room).us + plan_tiles_bf16(rows, groups, width, ff, room).us + 8.0f + glu;
    return direct < (groups > 1 ? 0.95f : plain ? 0.9f : 0.85f) * tiles;
}

// The launch in front of a product can leave its rows as bfloat16, for the direct form, or as F32, for ntk_dense.  Of 450 sizes each (9 .. 1000 rows, 512 .. 4096 outputs, 256 .. 4096 inputs; a norm, a
// gate, a norm and gate in front, both launches in a graph) always direct was behind by more than 2 % in 43, 62 and 68: fewer than eight chunks, which cost less than a direct tile's first requests
// (65 x 2048 x 256 7.2 us / 6.4 over F32 rows; many rows are ahead again, 1000 x 2048 x 256 by 15 %), and behind a gate, whose launch gains less, up to 1024 inputs that the tiles cut into pieces and
// this form does not (48 x 512 x 768 8.9 / 8.2, behind a norm 9.1 / 9.1).  So in none, at 0.81, 0.89 and 0.89 of the time over F32 rows: 150 x 1024 x 2048 12.5 / 15.9, 12 x 4096 x 4096 15.2 / 24.3.
int ntk_dense_direct_ahead(int T, int N, int K, int gate, size_t scratch_bytes) {
    if (!ntk_dense_direct_takes(NTK_DT_BF16, T, T, N, K)) return 0;
    const long long room = T > 65535 ? 0 : (long long)(scratch_bytes / sizeof(float));
    const TilePlan q = plan_direct_bf16(T, 1, N, K, room), p = plan_tiles_bf16(T, 1, N, K, room);
    if (K < 512) return T >= 500 || q.us < p.us + 2.5f;
    return !(gate && K < 1024 && p.splits > 1 && q.splits == 1 && q.us >= p.us + 1.15f);
}
int ntk_dense_direct_plan(int rows, int groups, int N, int K, long long room, int* plan) {
    if (!plan) return NTK_E_NULL;
    if (rows <= 0 || groups <= 0 || N <= 0 || K <= 0) return NTK_E_SHAPE;
    const TilePlan p = plan_direct_bf16(rows, groups, N, K, room);
    tell_plan(kFormsBf16[p.form], p, plan);
    return NTK_OK;
}
int ntk_dense_direct(const ntk_dense_desc* d, const ntk_direct_desc* e, void* stream) {
    if (!d || !e || !d->W || !e->x16 || (!e->y16 && !d->Y)) return NTK_E_NULL;
    if (!ntk_dense_direct_takes(d->wdtype, d->T, e->x16_rows, d->N, d->K)) return d->T == 0 ? NTK_OK : NTK_E_SHAPE;
    const bool glu = d->glu_ff > 0, bf = d->wdtype == NTK_DT_BF16;
    const int es = bf ? 2 : 4;
    if (e->ldx16 < d->K || e->ldx16 % (16 / es) || d->wstride % (16 / es) || (long long)e->x16_rows * e->ldx16 * es >= 1LL << 32 || (!bf && e->y16)) return NTK_E_SHAPE;
    if (((uintptr_t)e->x16 | (uintptr_t)d->W) & 15) return NTK_E_ALIGN;
    if (e->y16 ? (e->ldy16 < (glu ? d->glu_ff : d->N) || d->accumulate) : (d->ldy < (glu ? d->glu_ff : d->N) || (glu && d->accumulate))) return NTK_E_SHAPE;
    if ((glu && (d->N != 2 * d->glu_ff || d->act)) || d->norm_w || d->add_y || d->full_x) return NTK_E_SHAPE;
    if ((d->offsets && d->G <= 0) || (d->rows && d->row_div <= 0) || (!d->rows && e->x16_rows < d->T)) return NTK_E_SHAPE;
    if ((d->act != NTK_ACT_NONE && d->act != NTK_ACT_RELU2) || (d->act && d->accumulate)) return NTK_E_SHAPE;
    const int G = d->offsets ? d->G : 1;
    DirectArgs a{};
    TileArgs& t = a.t;
    t.Y = d->Y; t.ldy = d->ldy; t.W = d->W; t.wstride = d->wstride; t.offsets = d->offsets; t.G = G; t.rows = d->rows; t.row_div = d->rows ? d->row_div : 1;
    t.T = d->T; t.N = d->N; t.K = d->K; t.accumulate = d->accumulate; t.act = d->act; t.part = d->scratch;
    a.X16 = e->x16; a.x_row = (uint32_t)e->ldx16 * es; a.Y16 = (uint16_t*)e->y16; a.ldy16 = e->ldy16;
    // (no pieces for grouped rows: rows that belong to no group stay untouched)
    const long long room = d->scratch && !((uintptr_t)d->scratch & 15) && !d->offsets && !e->y16 && !glu && d->T <= 65535 ? (long long)(d->scratch_bytes / sizeof(float)) : 0;
    hipStream_t s = resolve_stream(stream);
    if (glu) {
        a.glu_ff = d->glu_ff; a.up_at = (uint32_t)d->glu_ff * (uint32_t)d->K * es; a.limit = d->glu_limit; a.alpha = d->glu_alpha; a.up_offset = d->glu_up_offset; a.cubic = d->glu_cubic;
    }
    if (!bf) {
        if (glu) launch_direct_f32<kGluClipped>(a, G, room, s);
        else launch_direct_f32<kGluNone>(a, G, room, s);
        return last_launch_status();
    }
    const TilePlan p = plan_direct_bf16(d->T, G, d->N, d->K, room);
    if (glu) launch_direct_bf16<kGluClipped>(a, p, s);
    else launch_direct_bf16<kGluNone>(a, p, s);
    return last_launch_status();
}

static int dense_with(const ntk_dense_desc* d, float cap, void* stream);
int ntk_dense(const ntk_dense_desc* d, void* stream) { return dense_with(d, 0.0f, stream); }
int ntk_dense_capped(const ntk_dense_desc* d, float cap, void* stream) {
    if (!d) return NTK_E_NULL;
    if (!(cap > 0.0f) || d->act || d->accumulate || d->glu_ff > 0) return NTK_E_SHAPE;
    const bool inside = d->T <= kGemvRows;              // (a launch of 4.6 us less behind the head of a decoded token)
    const int st = dense_with(d, inside ? cap : 0.0f, stream);
    return st != NTK_OK || inside ? st : ntk_softcap_rows(d->Y, d->ldy, cap, d->T, d->N, stream);
}
static int dense_with(const ntk_dense_desc* d, float cap, void* stream) {
    if (!d || !d->Y || !d->X || !d->W) return NTK_E_NULL;
    if (d->wdtype != NTK_DT_BF16 && d->wdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (d->T < 0 || d->N <= 0 || d->K <= 0 || d->ldx < d->K || d->ldy < (d->glu_ff > 0 ? d->glu_ff : d->N)) return NTK_E_SHAPE;
    if (d->offsets && d->G <= 0) return NTK_E_SHAPE;
    if (d->rows && d->row_div <= 0) return NTK_E_SHAPE;
    if (d->glu_ff > 0 && (d->T > kGemvRows || d->N != 2 * d->glu_ff || d->accumulate)) return NTK_E_SHAPE;
    if (d->norm_w && d->T > kGemvRows) return NTK_E_SHAPE;
    if ((d->act != NTK_ACT_NONE && d->act != NTK_ACT_RELU2) || (d->act && (d->accumulate || d->glu_ff > 0))) return NTK_E_SHAPE;
    if (d->add_y && (!d->add_w || !d->x_out)) return NTK_E_NULL;
    if (d->add_y && (d->T > kGemvRows || d->rows || d->offsets || d->ld_add < d->K || d->ldxo < d->K || d->x_out == d->X || d->x_out == d->add_y)) return NTK_E_SHAPE;
    if (d->T == 0) return NTK_OK;
    const int G = d->offsets ? d->G : 1;
    DenseArgs a{d->Y, d->ldy, d->X, d->ldx, d->W, d->wstride, d->offsets, d->rows, d->rows ? d->row_div : 1, d->T, d->N, d->K, d->accumulate, G, 0, 0, 0, 0.0f, 0.0f, 0.0f, 0.0f, nullptr, 0.0f, 0.0f, d->act, nullptr, 0, nullptr, 0.0f, 0.0f, nullptr, 0};
    hipStream_t s = resolve_stream(stream);
    if (d->T <= kGemvRows) {
        if (d->K > kGemvInputs) return NTK_E_SHAPE;
        a.glu_ff = d->glu_ff; a.glu_limit = d->glu_limit; a.glu_alpha = d->glu_alpha; a.glu_up_offset = d->glu_up_offset; a.glu_cubic = d->glu_cubic;
        a.norm_w = d->norm_w; a.norm_eps = d->norm_eps; a.norm_offset = d->norm_offset;
        if (cap > 0.0f) { a.act = kActCap; a.glu_limit = cap; }
        a.vec = (d->K % 8 == 0) && !((uintptr_t)d->W & 15) && !((d->wstride * (d->wdtype == NTK_DT_BF16 ? 2 : 4)) & 15);
        a.xvec = (d->K % 4 == 0) && (d->ldx % 4 == 0) && !((uintptr_t)d->X & 15) && !((uintptr_t)d->norm_w & 15);
        if (d->add_y) {
            a.add_y = d->add_y; a.ld_add = d->ld_add; a.add_w = d->add_w; a.add_eps = d->add_eps; a.add_mult = d->add_mult; a.x_out = d->x_out; a.ldxo = d->ldxo;
            a.xvec = a.xvec && (d->ld_add % 4 == 0) && (d->ldxo % 4 == 0) && !(((uintptr_t)d->add_y | (uintptr_t)d->add_w | (uintptr_t)d->x_out) & 15);
            if (d->wdtype == NTK_DT_BF16) launch_gemv<uint16_t, true>(a, d->T, s);
            else launch_gemv<float, true>(a, d->T, s);
            return last_launch_status();
        }
        if (d->wdtype == NTK_DT_BF16) launch_gemv<uint16_t, false>(a, d->T, s);
        else launch_gemv<float, false>(a, d->T, s);
        return last_launch_status();
    }
    const bool bf = d->wdtype == NTK_DT_BF16;
    TileArgs t{};
    t.Y = d->Y; t.ldy = d->ldy; t.X = d->X; t.ldx = d->ldx; t.W = d->W; t.wstride = d->wstride; t.offsets = d->offsets; t.G = G; t.rows = d->rows; t.row_div = a.row_div;
    t.T = d->T; t.N = d->N; t.K = d->K; t.accumulate = d->accumulate; t.act = d->act; t.part = d->scratch;
    const int align = bf ? 8 : 4;
    const bool vec = (d->K % align == 0) && d->K < 1 << 24 && (d->ldx % 4 == 0) && !((uintptr_t)d->X & 15) && !((uintptr_t)d->W & 15) && (d->wstride % align == 0);
    if (bf && d->full_x) {                 // (a few tokens' rows: one small tile)
        if (vec) launch_tiles<TileBf16x3, 32, 64, 2, 2, 2, true>(t, 1, s);
        else launch_tiles<TileBf16x3, 32, 64, 2, 2, 2, false>(t, 1, s);
        return last_launch_status();
    }
    if (!vec) {
        // odd sizes and addresses, element by element into the tiles.  bf16: from three 64 x 64 tiles a CU on, twice the tile -- fewer element-wise readings of either operand: us at
        // K = 2047 with 64 x 64 / 128 x 128: 1024 x 7488 556 / 346, 400 x 7488 (819 tiles) 269 / 201, 800 x 2048 (416) 147 / 197, 1024 x 2048 (512) 156 / 199; in 16
        // groups of 2815 outputs 1600 rows 369 / 332, 600 rows 187 / 280
        const int row_tiles = G > 1 ? d->T / 64 + (G + 1) / 2 : (d->T + 63) / 64;
        if (bf && (long long)row_tiles * ((d->N + 63) / 64) > 768) launch_tiles<TileBf16, 128, 128, 1, 4, 2, false>(t, 1, s);
        else if (bf) launch_tiles<TileBf16, 64, 64, 2, 2, 2, false>(t, 1, s);
        else launch_tiles<TileF32, 64, 64, 2, 2, 2, false>(t, 1, s);
        return last_launch_status();
    }
    // (no pieces for grouped rows: rows that belong to no group stay untouched)
    const long long room = d->scratch && !((uintptr_t)d->scratch & 15) && !d->offsets && d->T <= 65535 ? (long long)(d->scratch_bytes / sizeof(float)) : 0;
    if (bf) {
        // (a launch that rounds the activations first, where the product over them gains more than that launch takes: rows K 16-bit values apart in the scratch, pieces behind them)
        const long long image = ((long long)d->T * d->K * 2 + 15) & ~15LL;
        const bool direct = d->scratch && !((uintptr_t)d->scratch & 15) && !d->rows && (long long)d->scratch_bytes >= image && ntk_dense_direct_takes(d->wdtype, d->T, d->T, d->N, d->K);
        const TilePlan p = plan_tiles_bf16(d->T, G, d->N, d->K, room);
        if (direct) {
            const long long left = d->offsets || d->T > 65535 ? 0 : ((long long)d->scratch_bytes - image) / (long long)sizeof(float);
            const TilePlan q = plan_direct_bf16(d->T, G, d->N, d->K, left);
            // (p.us is the chunks' time alone.  With a twentieth in hand for the estimates none of 894 sizes of one matrix is behind the tiles by more than 1 %; in groups, whose tiles are
            // an average, by none of 2918 with 0.7 of the tiles' time -- at equal estimates 183 were, by up to a third: 500 rows in 4 groups of 256 x 1024 8.7 and 11.7 us)
            if (q.us + kRoundUs + (float)d->T * d->K * 6.0f / kRoundRate < (G > 1 ? 0.7f : 0.95f) * (p.us + 4.0f)) {
                const int st = ntk_round_rows(d->scratch, d->K, d->X, d->ldx, d->T, d->K, stream);
                if (st != NTK_OK) return st;
                DirectArgs a16{};
                a16.t = t;
                a16.t.part = (float*)((char*)d->scratch + image);
                a16.X16 = d->scratch; a16.x_row = (uint32_t)d->K * 2;
                launch_direct_bf16<kGluNone>(a16, q, s);
                return last_launch_status();
            }
        }
        if (p.form == 0) launch_tiles<TileBf16, 128, 128, 1, 4, 2, true>(t, p.splits, s);
        else if (p.form == 1) launch_tiles<TileBf16, 64, 128, 2, 2, 4, true>(t, p.splits, s);
        else if (p.form == 2) launch_tiles<TileBf16, 64, 64, 2, 2, 2, true>(t, p.splits, s);
        else launch_tiles<TileBf16, 32, 64, 2, 2, 2, true>(t, p.splits, s);
    } else {
        if (!d->rows && d->ldx % 4 == 0 && d->wstride % 4 == 0 && ntk_dense_direct_takes(d->wdtype, d->T, d->T, d->N, d->K) && (long long)d->T * d->ldx * 4 < 1LL << 32) {
            DirectArgs a32{};
            a32.t = t; a32.X16 = d->X; a32.x_row = (uint32_t)d->ldx * 4;
            launch_direct_f32<kGluNone>(a32, G, room, s);
            return last_launch_status();
        }
        static const TileForm forms[] = {{64, 64, 32, 0.78f, 0.70f}, {32, 64, 32, 0.52f, 0.36f}};
        const TilePlan p = plan_tiles(forms, 2, d->T, G, d->N, d->K, room);
        if (p.form == 0) launch_tiles<TileF32, 64, 64, 2, 2, 2, true>(t, p.splits, s);
        else launch_tiles<TileF32, 32, 64, 2, 2, 2, true>(t, p.splits, s);
    }
    return last_launch_status();
}

int ntk_moe_few(const ntk_moe_few_desc* d, void* stream) {
    if (!d || !d->out || !d->h || !d->ids || !d->wts || !d->up || !d->down || !d->mid || (d->shared_ff > 0 && (!d->shared_up || !d->shared_down))) return NTK_E_NULL;
    if (d->wdtype != NTK_DT_BF16 && d->wdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if ((d->act != NTK_ACT_NONE && d->act != NTK_ACT_RELU2) || (d->glu && d->act)) return NTK_E_SHAPE;
    if (d->mix && d->ld_mix < d->n) return NTK_E_SHAPE;
    if (d->T < 0 || d->T > kGemvRows || d->n <= 0 || d->top <= 0 || d->experts <= 0 || d->ff <= 0 || d->shared_ff < 0 || d->ldo < d->n || d->ldh < d->n) return NTK_E_SHAPE;
    if ((long long)d->top * d->ff + d->shared_ff > NTK_MOE_FEW_MID || d->n > NTK_MOE_FEW_MID) return NTK_E_SHAPE;
    if (d->T == 0) return NTK_OK;
    MoeFewArgs a{d->out, d->ldo, d->h, d->ldh, d->ids, d->wts, d->top, d->experts, d->up, d->down, d->shared_up, d->shared_down, d->ff, d->shared_ff, d->sgate, d->act, d->mid, d->n, 0};
    a.limit = d->glu_limit; a.shared_limit = d->shared_limit; a.alpha = d->glu_alpha; a.up_offset = d->glu_up_offset; a.mix = d->mix; a.ld_mix = d->ld_mix;
    a.vec = d->n % 8 == 0 && d->ff % 8 == 0 && d->shared_ff % 8 == 0 && d->ldh % 4 == 0 &&
            !(((uintptr_t)d->h | (uintptr_t)d->mid | (uintptr_t)d->up | (uintptr_t)d->down | (uintptr_t)d->shared_up | (uintptr_t)d->shared_down) & 15);
    static bool raised = false;     // (idempotent: a race sets the same attributes twice)
    if (!raised) {
        const void* fn[] = {(const void*)moe_few_up_kernel<uint16_t, 2, false>, (const void*)moe_few_up_kernel<float, 2, false>, (const void*)moe_few_up_kernel<uint16_t, 2, true>,
                            (const void*)moe_few_up_kernel<float, 2, true>};
        for (const void* f : fn) NTK_HIP_TRY(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, NTK_MOE_FEW_MID * 4));
        raised = true;
    }
    if (d->wdtype == NTK_DT_BF16) launch_moe_few<uint16_t>(a, d->T, d->glu != 0, resolve_stream(stream));
    else launch_moe_few<float>(a, d->T, d->glu != 0, resolve_stream(stream));
    return last_launch_status();
}

int ntk_dense_few_rows(void) { return kGemvRows; }
int ntk_dense_few_inputs(void) { return ntk::kGemvInputs; }

int ntk_dense_linear(float* Y, int ldy, const float* X, int ldx, const void* W, int wdtype, int T, int N, int K, int accumulate, void* stream) {
    ntk_dense_desc d{};
    d.Y = Y; d.ldy = ldy; d.X = X; d.ldx = ldx; d.W = W; d.wstride = 0; d.wdtype = wdtype; d.offsets = nullptr; d.G = 1; d.rows = nullptr; d.row_div = 1;
    d.T = T; d.N = N; d.K = K; d.accumulate = accumulate;
    return ntk_dense(&d, stream);
}
