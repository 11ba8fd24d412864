// layer_ops.hip -- the small F32 operators around the products of the layer-list families: dense embedding rows, RMS norms whose weight is stored
// plain or around zero (two outputs from one pass over x: the two norms of a parallel layer read the same residual row), layer norms with weight and
// bias (also added onto the stream), the short causal convolution that is added to a sublayer's input (with its carried inputs), the polynomial
// activation with unit-norm terms, the gated RMS norm, row concatenation, sigmoid gates, the residual sum.  Everything is F32; one workgroup per row
// where a row is reduced.
#include "common.hip.h"
#include "../../include/ntk_layers.h"

namespace ntk {

template <typename TT>
__global__ __launch_bounds__(256) void embed_dense_kernel(float* out, const TT* table, const int* tokens, int vocab, int width, float scale) {
    const int t = blockIdx.x, tok = tokens[t];
    float* o = out + (long long)t * width;
    const bool ok = tok >= 0 && tok < vocab;
    const TT* row = table + (long long)(ok ? tok : 0) * width;
    for (int i = threadIdx.x; i < width; i += 256) {
        float v = 0.0f;
        if (ok) {
            if constexpr (sizeof(TT) == 2) v = __uint_as_float((uint32_t)row[i] << 16); else v = row[i];
        }
        o[i] = v * scale;
    }
}

// ... four entries a thread (width % 4 == 0, aligned); tokens NULL: one token, given with the launch.  us, one row of 2048 / 1024 rows: 5.7 / 8.1 a workgroup a row above, 2.5 / 4.5 so
template <typename TT>
__global__ __launch_bounds__(256) void embed_dense_wide_kernel(float* out, const TT* table, const int* tokens, int token, int vocab, int width, float scale) {
    const int t = blockIdx.y, i = 4 * ((int)blockIdx.x * 256 + (int)threadIdx.x), tok = tokens ? tokens[t] : token;
    if (i >= width) return;
    float4 v{0.0f, 0.0f, 0.0f, 0.0f};
    if (tok >= 0 && tok < vocab) {
        const TT* row = table + (long long)tok * width + i;
        if constexpr (sizeof(TT) == 2) {
            const uint2 b = *reinterpret_cast<const uint2*>(row);
            v = float4{__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xFFFF0000u), __uint_as_float(b.y << 16), __uint_as_float(b.y & 0xFFFF0000u)};
        } else v = *reinterpret_cast<const float4*>(row);
    }
    *reinterpret_cast<float4*>(out + (long long)t * width + i) = float4{v.x * scale, v.y * scale, v.z * scale, v.w * scale};
}

template <typename TT> __device__ __forceinline__ float table_value(const TT* row, int i) {
    if constexpr (sizeof(TT) == 2) return __uint_as_float((uint32_t)row[i] << 16); else return row[i];
}
// the token's row plus a row picked by the token and the one before it
template <typename TT>
__global__ __launch_bounds__(256) void embed_bigram_kernel(float* out, const TT* table, const TT* bigram, const int* tokens, int prev, int pos0, int vocab, int width,
                                                           float scale, int buckets, long long mul_prev, long long mul_cur) {
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x, tok = tokens[t];
    if (i >= width) return;
    const bool ok = tok >= 0 && tok < vocab;
    long long r = buckets;                                   // a sequence's first token
    if (pos0 + t > 0) {
        r = ((long long)(t > 0 ? tokens[t - 1] : prev) * mul_prev + (long long)tok * mul_cur) % buckets;
        if (r < 0) r += buckets;
    }
    const float e = table_value(table + (long long)(ok ? tok : 0) * width, i), b = table_value(bigram + r * width, i);
    out[(long long)t * width + i] = fmaf(ok ? e : 0.0f, scale, b);
}

// a thread owns the pair (2i, 2i + 1): sin and cos of one angle, formed in double
template <typename TT>
__global__ __launch_bounds__(256) void embed_sinusoid_kernel(float* out, const TT* table, const int* tokens, int vocab, int width, float scale, const double* freq, int pos0) {
    const int t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x, tok = tokens[t];
    if (2 * i >= width) return;
    const bool ok = tok >= 0 && tok < vocab;
    const TT* row = table + (long long)(ok ? tok : 0) * width;
    float* o = out + (long long)t * width;
    double sn, cs;
    sincos((double)(pos0 + t) * freq[i], &sn, &cs);
    o[2 * i] = fmaf(ok ? table_value(row, 2 * i) : 0.0f, scale, (float)sn);
    if (2 * i + 1 < width) o[2 * i + 1] = fmaf(ok ? table_value(row, 2 * i + 1) : 0.0f, scale, (float)cs);
}

__global__ __launch_bounds__(256) void rmsnorm_offset_kernel(float* y1, const float* w1, float* y2, const float* w2, int ldy, const float* x, int ldx, int n,
                                                             float eps, float offset) {
    __shared__ float red[16];
    const float* xr = x + (long long)blockIdx.x * ldx;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) ss = fmaf(xr[i], xr[i], ss);
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)n + eps);
    float* o1 = y1 + (long long)blockIdx.x * ldy;
    float* o2 = y2 ? y2 + (long long)blockIdx.x * ldy : nullptr;
    for (int i = threadIdx.x; i < n; i += 256) {
        const float u = xr[i] * inv;
        o1[i] = u * (offset + w1[i]);
        if (o2) o2[i] = u * (offset + w2[i]);
    }
}

// One workgroup a row of up to 4096 entries (a multiple of four, on 16 bytes): the row and everything it is combined with are requested before the first sum and cross memory
// once; results leave as F32, as bfloat16 (for a product that would round them at its input) or both.  Bound by the bytes of the rows; 1024 rows of 2048, rows_seam: 10.9 us with
// one value a request and F32 results, 6.6 so; rows_norm with two results 10.5, 6.8 with a third.
__device__ __forceinline__ uint2 pack4_bf16(const float4 v) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const b2 lo = __builtin_convertvector(f2{v.x, v.y}, b2), hi = __builtin_convertvector(f2{v.z, v.w}, b2);
    uint2 u;
    __builtin_memcpy(&u.x, &lo, 4);
    __builtin_memcpy(&u.y, &hi, 4);
    return u;
}
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float square4(const float4 v, float s) { return fmaf(v.w, v.w, fmaf(v.z, v.z, fmaf(v.y, v.y, fmaf(v.x, v.x, s)))); }
constexpr int kRowKeep = 4;       // float4s of a thread

__global__ __launch_bounds__(256) void rows_seam_kernel(uint16_t* h, float* x, int ldx, const float* add_y, int ldy, const float* add_w, float mult, const float* w, int n, float eps) {
    __shared__ float red[16];
    float* xr = x + (long long)blockIdx.x * ldx;
    const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    float4 v[kRowKeep], y[kRowKeep], aw[kRowKeep], nw[kRowKeep];
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) {
        const int i = 4 * (threadIdx.x + 256 * k);
        const bool in = i < n;
        if (add_y) { y[k] = in ? load4(add_y + (long long)blockIdx.x * ldy + i) : zero; aw[k] = in ? load4(add_w + i) : zero; }
        v[k] = in ? load4(xr + i) : zero;
        nw[k] = in ? load4(w + i) : zero;
    }
    if (add_y) {
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < kRowKeep; ++k) ss = square4(y[k], ss);
        const float inv = mult / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
        for (int k = 0; k < kRowKeep; ++k) {
            const int i = 4 * (threadIdx.x + 256 * k);
            v[k] = float4{fmaf(y[k].x * inv, aw[k].x, v[k].x), fmaf(y[k].y * inv, aw[k].y, v[k].y), fmaf(y[k].z * inv, aw[k].z, v[k].z), fmaf(y[k].w * inv, aw[k].w, v[k].w)};
            if (i < n) *reinterpret_cast<float4*>(xr + i) = v[k];
        }
    }
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) ss = square4(v[k], ss);
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) {
        const int i = 4 * (threadIdx.x + 256 * k);
        if (i < n) *reinterpret_cast<uint2*>(h + (long long)blockIdx.x * n + i) = pack4_bf16(float4{v[k].x * inv * nw[k].x, v[k].y * inv * nw[k].y, v[k].z * inv * nw[k].z, v[k].w * inv * nw[k].w});
    }
}

struct NormOut { float* y; uint16_t* y16; const float* w; };
__global__ __launch_bounds__(256) void rows_norm_kernel(const NormOut a, const NormOut b, int ldy, const float* x, int ldx, int n, float eps, float offset) {
    __shared__ float red[16];
    const float* xr = x + (long long)blockIdx.x * ldx;
    const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    float4 v[kRowKeep], wa[kRowKeep], wb[kRowKeep];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) {
        const int i = 4 * (threadIdx.x + 256 * k);
        v[k] = i < n ? load4(xr + i) : zero;
        wa[k] = i < n ? load4(a.w + i) : zero;
        wb[k] = b.w && i < n ? load4(b.w + i) : zero;
    }
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) ss = square4(v[k], ss);
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
    for (int k = 0; k < kRowKeep; ++k) {
        const int i = 4 * (threadIdx.x + 256 * k);
        if (i >= n) continue;
        const float4 u{v[k].x * inv, v[k].y * inv, v[k].z * inv, v[k].w * inv};
        auto put = [&](const NormOut& o, const float4 w) {
            const float4 r{u.x * (offset + w.x), u.y * (offset + w.y), u.z * (offset + w.z), u.w * (offset + w.w)};
            if (o.y) *reinterpret_cast<float4*>(o.y + (long long)blockIdx.x * ldy + i) = r;
            if (o.y16) *reinterpret_cast<uint2*>(o.y16 + (long long)blockIdx.x * n + i) = pack4_bf16(r);
        };
        put(a, wa[k]);
        if (b.w) put(b, wb[k]);
    }
}

__global__ void concat_rows_kernel(float* out, const float* a, const float* b, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * n) return;
    out[t * 2 * n + i] = i < n ? a[t * n + i] : b[t * n + (i - n)];
}

__global__ void sigmoid_gate_kernel(float* y, int ldy, const float* g, int ldg, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[t * ldy + i] *= 1.0f / (1.0f + expf(-g[t * ldg + i]));
}

__global__ void rows_copy_kernel(float* dst, const float* src, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ void residual_add_kernel(float* x, const float* a, const float* b, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float s = a[i];
    if (b) s += b[i];
    x[i] += s;
}

__global__ void scale_kernel(float* x, long long n, float s) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] *= s;
}

// mean first, then the mean of the squared deviations, then the outputs.  A thread keeps its first LN_KEEP entries (i = tid + 256 k) in registers -- rows up to
// 4096 wide are read once --; what lies beyond is read again (it sits in the cache).  Returns through (mean, inv); `emit(i, normed value)` writes.
// Workgroups of NT threads: 256 where a launch has many rows, 1024 where it has few (decoding: a row's entries are then spread over four times the threads,
// whose loads are in flight together -- a thread's own entries follow each other through load, use and store).
template <int NT, typename Emit>
__device__ __forceinline__ void layernorm_row(const float* xr, const float* w, const float* b, int n, float eps, float* red, Emit emit) {
    constexpr int KEEP = 4096 / NT;
    float v[KEEP], wv[KEEP], bv[KEEP];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
        const int i = threadIdx.x + NT * k;
        v[k] = i < n ? xr[i] : 0.0f;
        wv[k] = i < n ? w[i] : 0.0f;
        bv[k] = i < n && b ? b[i] : 0.0f;
        s += v[k];
    }
    for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) s += xr[i];
    const float mean = block_sum(s, red) / (float)n;
    float q = 0.0f;
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
        const float d = v[k] - mean;
        if ((int)threadIdx.x + NT * k < n) q = fmaf(d, d, q);
    }
    for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) { const float d = xr[i] - mean; q = fmaf(d, d, q); }
    const float inv = 1.0f / sqrtf(block_sum(q, red) / (float)n + eps);
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
        const int i = threadIdx.x + NT * k;
        if (i < n) emit(i, (v[k] - mean) * inv * wv[k] + bv[k]);
    }
    for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) emit(i, (xr[i] - mean) * inv * w[i] + (b ? b[i] : 0.0f));
}

template <int NT>
__global__ __launch_bounds__(NT) void layernorm_kernel(float* y, int ldy, const float* x, int ldx, const float* w, const float* b, int n, float eps, int accumulate) {
    __shared__ float red[16];
    float* yr = y + (long long)blockIdx.x * ldy;
    if (accumulate) layernorm_row<NT>(x + (long long)blockIdx.x * ldx, w, b, n, eps, red, [&](int i, float o) { yr[i] += o; });
    else layernorm_row<NT>(x + (long long)blockIdx.x * ldx, w, b, n, eps, red, [&](int i, float o) { yr[i] = o; });
}

// rows 0 .. taps-2: the carried inputs (zeros before the sequence's start); rows taps-1 ..: the layer norm of the portion's tokens.  With add_y the stream row
// first takes the sublayer output that is still owed to it, x[t] += layer norm of add_y[t] (weights add_w / add_b): the norm after one sublayer and the norm
// before the next in one pass over the row (a thread reads back only what it wrote itself).
__global__ __launch_bounds__(256) void layernorm_history_kernel(float* hist, float* x, int ldx, const float* w, const float* b, const float* state, int taps,
                                                                int pos0, int n, float eps, const float* add_y, int ldy, const float* add_w, const float* add_b) {
    __shared__ float red[16];
    const int r = blockIdx.x;
    float* o = hist + (long long)r * n;
    if (r < taps - 1) {
        const bool before = pos0 - (taps - 1) + r < 0;
        for (int i = threadIdx.x; i < n; i += 256) o[i] = before ? 0.0f : state[(long long)r * n + i];
        return;
    }
    float* xr = x + (long long)(r - (taps - 1)) * ldx;
    if (add_y) layernorm_row<256>(add_y + (long long)(r - (taps - 1)) * ldy, add_w, add_b, n, eps, red, [&](int i, float v) { xr[i] += v; });
    layernorm_row<256>(xr, w, b, n, eps, red, [&](int i, float v) { o[i] = v; });
}

// one token (decoding), one workgroup: the owed sublayer output onto the stream, the norm, the convolution over the carried inputs and their shift -- every
// channel's history belongs to the thread that owns the channel.  Same sums in the same order as the two launches of a longer portion.
constexpr int kStepThreads = 1024;
__global__ __launch_bounds__(kStepThreads) void sandwich_step_kernel(float* out, float* x, const float* w, const float* b, const float* canon, float* state, int taps, int pos0,
                                                            int n, float eps, const float* add_y, const float* add_w, const float* add_b) {
    __shared__ float red[16];
    if (add_y) layernorm_row<kStepThreads>(add_y, add_w, add_b, n, eps, red, [&](int i, float v) { x[i] += v; });
    layernorm_row<kStepThreads>(x, w, b, n, eps, red, [&](int i, float h) {
        const float* cw = canon + (long long)i * taps;
        float s = 0.0f;
        for (int j = 0; j < taps - 1; ++j) {
            const float hj = pos0 - (taps - 1) + j >= 0 ? state[(long long)j * n + i] : 0.0f;
            s = fmaf(cw[j], hj, s);
            if (j > 0) state[(long long)(j - 1) * n + i] = hj;
        }
        s = fmaf(cw[taps - 1], h, s);
        if (taps > 1) state[(long long)(taps - 2) * n + i] = h;
        out[i] = h + s;
    });
}

// blocks y < T: out[y] = hist[taps-1+y] + sum_j w[:, j] * hist[y+j] (j ascending); blocks y >= T: the carried rows for the next portion
__global__ void causal_conv_mix_kernel(float* out, int ldo, const float* hist, const float* w, float* state, int taps, int T, int n) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (c >= n) return;
    if (y >= T) { state[(long long)(y - T) * n + c] = hist[(long long)y * n + c]; return; }
    float s = 0.0f;
    for (int j = 0; j < taps; ++j) s = fmaf(w[(long long)c * taps + j], hist[(long long)(y + j) * n + c], s);
    out[(long long)y * ldo + c] = hist[(long long)(y + taps - 1) * n + c] + s;
}

__global__ __launch_bounds__(1024) void polynorm_kernel(float* y, int ldy, const float* z, int ldz, const float* coef, int n, float eps) {
    __shared__ float red[16];
    const float* zr = z + (long long)blockIdx.x * ldz;
    float s2 = 0.0f, s4 = 0.0f, s6 = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = zr[i], v2 = v * v, v3 = v2 * v;
        s2 += v2; s4 = fmaf(v2, v2, s4); s6 = fmaf(v3, v3, s6);
    }
    s2 = block_sum(s2, red); s4 = block_sum(s4, red); s6 = block_sum(s6, red);
    const float i1 = coef[0] / sqrtf(s2 / (float)n + eps), i2 = coef[1] / sqrtf(s4 / (float)n + eps), i3 = coef[2] / sqrtf(s6 / (float)n + eps), e = coef[3];
    float* o = y + (long long)blockIdx.x * ldy;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = zr[i], v2 = v * v, v3 = v2 * v;
        o[i] = i1 * v + i2 * v2 + i3 * v3 + e;
    }
}

__global__ __launch_bounds__(1024) void gated_rmsnorm_kernel(float* y, int ldy, const float* x, int ldx, const float* w, const float* g, int ldg, int n, float eps) {
    __shared__ float red[16];
    const float* xr = x + (long long)blockIdx.x * ldx;
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) ss = fmaf(xr[i], xr[i], ss);
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
    float* o = y + (long long)blockIdx.x * ldy;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float v = xr[i] * inv * w[i];
        if (g) v *= 1.0f / (1.0f + expf(-g[(long long)blockIdx.x * ldg + i]));
        o[i] = v;
    }
}

constexpr int kFewRows = 32;   // up to this many rows a row kernel runs workgroups of 1024 threads

// ---- what a pass takes from the host and leaves there: words as arguments of a launch, results by a launch's own stores into pinned memory.  A decoded token of 32000 logits spent 5 + 5 us
// on two copies of the runtime and waited for the stream twice (a copy into pageable memory is one more round trip of the host); so 2 + 4 and once.
struct Words { int v[32]; };
__global__ __launch_bounds__(64) void store_words_kernel(int* __restrict__ a, int na, int* __restrict__ b, int n, const Words w) {
    const int i = threadIdx.x;
    if (i >= n) return;
    if (i < na) a[i] = w.v[i];
    else b[i - na] = w.v[i];
}
// a piece a workgroup: its stores are out (system scope) in front of its word (there NULL: no words, the stream is waited for)
__global__ __launch_bounds__(256) void copy_out_pieces_kernel(uint32_t* __restrict__ out, const uint32_t* __restrict__ src, size_t words, int wide, unsigned* __restrict__ there, unsigned turn, int* __restrict__ bump) {
    const size_t at = (size_t)blockIdx.x * NTK_COPY_OUT_PIECE, end = min(words, at + NTK_COPY_OUT_PIECE);
    if (bump && blockIdx.x == 0 && threadIdx.x == 0) *bump += 1;
    if (wide && at + NTK_COPY_OUT_PIECE <= words) {
#pragma unroll
        for (int k = 0; k < NTK_COPY_OUT_PIECE / 1024; ++k) {
            const size_t i = at + 4 * (size_t)(threadIdx.x + 256 * k);
            *reinterpret_cast<uint4*>(out + i) = *reinterpret_cast<const uint4*>(src + i);
        }
    } else
        for (size_t i = at + threadIdx.x; i < end; i += 256) out[i] = src[i];
    if (!there) return;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(there + blockIdx.x, turn, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace ntk

using namespace ntk;

int ntk_store_words(int* a, int na, int* b, int nb, const int* values, void* stream) {
    if ((!a && na > 0) || (!b && nb > 0) || !values) return NTK_E_NULL;
    if (na < 0 || nb < 0 || na + nb > 32) return NTK_E_SHAPE;
    if (na + nb == 0) return NTK_OK;
    Words w{};
    for (int i = 0; i < na + nb; ++i) w.v[i] = values[i];
    hipLaunchKernelGGL(store_words_kernel, dim3(1), dim3(64), 0, resolve_stream(stream), a, na, b, na + nb, w);
    return last_launch_status();
}
int ntk_copy_out(void* pinned, const void* src, size_t size, void* stream) {
    if (!pinned || !src) return NTK_E_NULL;
    const uintptr_t at = (uintptr_t)pinned | (uintptr_t)src;
    if (size % 4 || size / 4 > (size_t)0x7FFFFFFF * 256) return NTK_E_SHAPE;
    if (at & 3) return NTK_E_ALIGN;
    if (size == 0) return NTK_OK;
    hipLaunchKernelGGL(copy_out_pieces_kernel, dim3((unsigned)ntk_copy_out_words(size / 4)), dim3(256), 0, resolve_stream(stream), static_cast<uint32_t*>(pinned), static_cast<const uint32_t*>(src),
                       size / 4, (int)((at & 15) == 0), static_cast<unsigned*>(nullptr), 0u, static_cast<int*>(nullptr));
    return last_launch_status();
}

size_t ntk_copy_out_words(size_t words) { return (words + NTK_COPY_OUT_PIECE - 1) / NTK_COPY_OUT_PIECE; }
int ntk_copy_out_pieces(void* pinned, const void* src, size_t words, unsigned* there, unsigned turn, int* bump, void* stream) {
    if (!pinned || !src || !there) return NTK_E_NULL;
    const uintptr_t at = (uintptr_t)pinned | (uintptr_t)src;
    if (words == 0 || words > (size_t)0x7FFFFFFF) return NTK_E_SHAPE;
    if ((at | (uintptr_t)there | (uintptr_t)bump) & 3) return NTK_E_ALIGN;
    hipLaunchKernelGGL(copy_out_pieces_kernel, dim3((unsigned)ntk_copy_out_words(words)), dim3(256), 0, resolve_stream(stream), static_cast<uint32_t*>(pinned), static_cast<const uint32_t*>(src),
                       words, (int)((at & 15) == 0), there, turn, bump);
    return last_launch_status();
}

int ntk_embed_dense(float* out, const void* table, int tdtype, const int* tokens, int T, int vocab, int width, void* stream) {
    return ntk_embed_dense_scaled(out, table, tdtype, tokens, T, vocab, width, 1.0f, stream);
}

static bool embed_wide(float* out, const void* table, int tdtype, const int* tokens, int token, int T, int vocab, int width, float scale, void* stream) {
    if (width % 4 || (((uintptr_t)out | (uintptr_t)table) & 15) || T > 65535) return false;
    const dim3 grid((width / 4 + 255) / 256, T);
    if (tdtype == NTK_DT_BF16) hipLaunchKernelGGL(embed_dense_wide_kernel<uint16_t>, grid, dim3(256), 0, resolve_stream(stream), out, (const uint16_t*)table, tokens, token, vocab, width, scale);
    else hipLaunchKernelGGL(embed_dense_wide_kernel<float>, grid, dim3(256), 0, resolve_stream(stream), out, (const float*)table, tokens, token, vocab, width, scale);
    return true;
}
int ntk_embed_token(float* out, const void* table, int tdtype, int token, int vocab, int width, float scale, void* stream) {
    if (!out || !table) return NTK_E_NULL;
    if (tdtype != NTK_DT_BF16 && tdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (vocab <= 0 || width <= 0) return NTK_E_SHAPE;
    return embed_wide(out, table, tdtype, nullptr, token, 1, vocab, width, scale, stream) ? last_launch_status() : NTK_E_ALIGN;
}

int ntk_embed_dense_scaled(float* out, const void* table, int tdtype, const int* tokens, int T, int vocab, int width, float scale, void* stream) {
    if (!out || !table || !tokens) return NTK_E_NULL;
    if (T < 0 || vocab <= 0 || width <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    if ((tdtype == NTK_DT_BF16 || tdtype == NTK_DT_F32) && embed_wide(out, table, tdtype, tokens, 0, T, vocab, width, scale, stream)) return last_launch_status();
    if (tdtype == NTK_DT_BF16) hipLaunchKernelGGL(embed_dense_kernel<uint16_t>, dim3(T), dim3(256), 0, resolve_stream(stream), out, (const uint16_t*)table, tokens, vocab, width, scale);
    else if (tdtype == NTK_DT_F32) hipLaunchKernelGGL(embed_dense_kernel<float>, dim3(T), dim3(256), 0, resolve_stream(stream), out, (const float*)table, tokens, vocab, width, scale);
    else return NTK_E_DTYPE;
    return last_launch_status();
}

int ntk_embed_bigram(float* out, const void* table, const void* bigram, int tdtype, const int* tokens, int prev, int pos0, int T, int vocab, int width, float scale,
                     int buckets, long long mul_prev, long long mul_cur, void* stream) {
    if (!out || !table || !bigram || !tokens) return NTK_E_NULL;
    if (tdtype != NTK_DT_BF16 && tdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (T < 0 || vocab <= 0 || width <= 0 || pos0 < 0 || buckets <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const dim3 grid((width + 255) / 256, T);
    if (tdtype == NTK_DT_BF16)
        hipLaunchKernelGGL(embed_bigram_kernel<uint16_t>, grid, dim3(256), 0, resolve_stream(stream), out, (const uint16_t*)table, (const uint16_t*)bigram, tokens, prev,
                           pos0, vocab, width, scale, buckets, mul_prev, mul_cur);
    else
        hipLaunchKernelGGL(embed_bigram_kernel<float>, grid, dim3(256), 0, resolve_stream(stream), out, (const float*)table, (const float*)bigram, tokens, prev, pos0,
                           vocab, width, scale, buckets, mul_prev, mul_cur);
    return last_launch_status();
}

int ntk_embed_sinusoid(float* out, const void* table, int tdtype, const int* tokens, int T, int vocab, int width, float scale, const double* freq, int pos0, void* stream) {
    if (!out || !table || !tokens || !freq) return NTK_E_NULL;
    if (tdtype != NTK_DT_BF16 && tdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (T < 0 || vocab <= 0 || width <= 0 || pos0 < 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const dim3 grid(((width + 1) / 2 + 255) / 256, T);
    if (tdtype == NTK_DT_BF16)
        hipLaunchKernelGGL(embed_sinusoid_kernel<uint16_t>, grid, dim3(256), 0, resolve_stream(stream), out, (const uint16_t*)table, tokens, vocab, width, scale, freq, pos0);
    else
        hipLaunchKernelGGL(embed_sinusoid_kernel<float>, grid, dim3(256), 0, resolve_stream(stream), out, (const float*)table, tokens, vocab, width, scale, freq, pos0);
    return last_launch_status();
}

int ntk_rmsnorm_offset(float* y1, const float* w1, float* y2, const float* w2, int ldy, const float* x, int ldx, int T, int n, float eps, float offset,
                       void* stream) {
    if (!y1 || !w1 || !x || (y2 && !w2)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(rmsnorm_offset_kernel, dim3(T), dim3(256), 0, resolve_stream(stream), y1, w1, y2, w2, ldy, x, ldx, n, eps, offset);
    return last_launch_status();
}

static bool whole_rows(int n, int ld1, int ld2, const void* p1, const void* p2, const void* p3) {      // what the kernels above take
    return n % 4 == 0 && n <= 4 * 256 * kRowKeep && ld1 % 4 == 0 && ld2 % 4 == 0 && !(((uintptr_t)p1 | (uintptr_t)p2 | (uintptr_t)p3) & 15);
}

int ntk_rmsnorm_offset_16(float* y1, void* y1_16, const float* w1, float* y2, void* y2_16, const float* w2, int ldy, const float* x, int ldx, int T, int n, float eps,
                          float offset, void* stream) {
    if ((!y1 && !y1_16) || !w1 || !x || ((y2 || y2_16) && !w2)) return NTK_E_NULL;
    const bool second = y2 || y2_16;
    if (T < 0 || n <= 0 || ((y1 || y2) && ldy < n) || ldx < n) return NTK_E_SHAPE;
    if (!whole_rows(n, y1 || y2 ? ldy : 0, ldx, y1, y2, x) || !whole_rows(n, 0, 0, w1, w2, nullptr) || (((uintptr_t)y1_16 | (uintptr_t)y2_16) & 7)) return NTK_E_ALIGN;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(rows_norm_kernel, dim3(T), dim3(256), 0, resolve_stream(stream), NormOut{y1, (uint16_t*)y1_16, w1}, NormOut{y2, (uint16_t*)y2_16, second ? w2 : nullptr}, ldy, x, ldx, n, eps,
                       offset);
    return last_launch_status();
}

int ntk_concat_rows(float* out, const float* a, const float* b, int T, int n, void* stream) {
    if (!out || !a || !b) return NTK_E_NULL;
    if (T < 0 || n <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(concat_rows_kernel, dim3((2 * n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), out, a, b, n);
    return last_launch_status();
}

int ntk_sigmoid_gate(float* y, int ldy, const float* g, int ldg, int T, int n, void* stream) {
    if (!y || !g) return NTK_E_NULL;
    if (T < 0 || n <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(sigmoid_gate_kernel, dim3((n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), y, ldy, g, ldg, n);
    return last_launch_status();
}

int ntk_rows_copy(float* dst, const float* src, long long n, void* stream) {
    if (!dst || !src) return NTK_E_NULL;
    if (n < 0 || n > (1ll << 38)) return NTK_E_SHAPE;
    if (n == 0) return NTK_OK;
    hipLaunchKernelGGL(rows_copy_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, resolve_stream(stream), dst, src, n);
    return last_launch_status();
}

int ntk_residual_add(float* x, const float* a, const float* b, int n, void* stream) {
    if (!x || !a) return NTK_E_NULL;
    if (n < 0) return NTK_E_SHAPE;
    if (n == 0) return NTK_OK;
    hipLaunchKernelGGL(residual_add_kernel, dim3((n + 255) / 256), dim3(256), 0, resolve_stream(stream), x, a, b, n);
    return last_launch_status();
}

int ntk_scale(float* x, long long n, float s, void* stream) {
    if (!x) return NTK_E_NULL;
    if (n < 0 || n > (1ll << 38)) return NTK_E_SHAPE;
    if (n == 0) return NTK_OK;
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, resolve_stream(stream), x, n, s);
    return last_launch_status();
}

int ntk_layernorm(float* y, int ldy, const float* x, int ldx, const float* w, const float* b, int T, int n, float eps, int accumulate, void* stream) {
    if (!y || !x || !w) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    if (T <= kFewRows) hipLaunchKernelGGL(layernorm_kernel<1024>, dim3(T), dim3(1024), 0, resolve_stream(stream), y, ldy, x, ldx, w, b, n, eps, accumulate);
    else hipLaunchKernelGGL(layernorm_kernel<256>, dim3(T), dim3(256), 0, resolve_stream(stream), y, ldy, x, ldx, w, b, n, eps, accumulate);
    return last_launch_status();
}

int ntk_layernorm_history(float* hist, const float* x, int ldx, const float* w, const float* b, const float* state, int taps, int pos0, int T, int n, float eps,
                          void* stream) {
    if (!hist || !x || !w || (taps > 1 && !state)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n || taps < 1 || pos0 < 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(layernorm_history_kernel, dim3(T + taps - 1), dim3(256), 0, resolve_stream(stream), hist, const_cast<float*>(x), ldx, w, b, state, taps, pos0, n,
                       eps, (const float*)nullptr, 0, (const float*)nullptr, (const float*)nullptr);
    return last_launch_status();
}

int ntk_sandwich_norm_conv(float* out, int ldo, float* x, int ldx, const float* add_y, int ldy, const float* add_w, const float* add_b, const float* w, const float* b,
                           const float* canon, float* state, float* hist, int taps, int pos0, int T, int n, float eps, void* stream) {
    if (!out || !x || !w || !canon || (taps > 1 && !state) || (add_y && !add_w)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n || ldo < n || (add_y && ldy < n) || taps < 1 || pos0 < 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipStream_t s = resolve_stream(stream);
    if (T == 1) {
        hipLaunchKernelGGL(sandwich_step_kernel, dim3(1), dim3(kStepThreads), 0, s, out, x, w, b, canon, state, taps, pos0, n, eps, add_y, add_w, add_b);
        return last_launch_status();
    }
    if (!hist) return NTK_E_NULL;
    hipLaunchKernelGGL(layernorm_history_kernel, dim3(T + taps - 1), dim3(256), 0, s, hist, x, ldx, w, b, (const float*)state, taps, pos0, n, eps, add_y, ldy, add_w, add_b);
    const int st = last_launch_status();
    if (st != NTK_OK) return st;
    return ntk_causal_conv_mix(out, ldo, hist, canon, state, taps, T, n, stream);
}

int ntk_causal_conv_mix(float* out, int ldo, const float* hist, const float* w, float* state, int taps, int T, int n, void* stream) {
    if (!out || !hist || !w || (taps > 1 && !state)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldo < n || taps < 1) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(causal_conv_mix_kernel, dim3((n + 255) / 256, T + taps - 1), dim3(256), 0, resolve_stream(stream), out, ldo, hist, w, state, taps, T, n);
    return last_launch_status();
}

int ntk_polynorm(float* y, int ldy, const float* z, int ldz, const float* coef, int T, int n, float eps, void* stream) {
    if (!y || !z || !coef) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldz < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(polynorm_kernel, dim3(T), dim3(T <= kFewRows ? 1024 : 256), 0, resolve_stream(stream), y, ldy, z, ldz, coef, n, eps);
    return last_launch_status();
}

int ntk_gated_rmsnorm(float* y, int ldy, const float* x, int ldx, const float* w, const float* g, int ldg, int T, int n, float eps, void* stream) {
    if (!y || !x || !w) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n || (g && ldg < n)) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(gated_rmsnorm_kernel, dim3(T), dim3(T <= kFewRows ? 1024 : 256), 0, resolve_stream(stream), y, ldy, x, ldx, w, g, ldg, n, eps);
    return last_launch_status();
}

// ---------------------------------------------------------------------------------------------------------------- layers with gated residuals
// The dynamic-tanh norm is element by element (no row sums), so it rides in whatever launch produces its input: the embedding (token row + position row),
// and the seam between sublayers (gated residual sum, the average over the layer results so far, the next norm).
namespace ntk {

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }

__global__ void dyt_kernel(float* y, int ldy, const float* x, int ldx, const float* w, const float* b, float alpha, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[t * ldy + i] = fmaf(tanhf(alpha * x[t * ldx + i]), w[i], b ? b[i] : 0.0f);
}

template <typename TT>
__global__ void embed_positions_kernel(float* out, float* copy, const TT* table, const TT* pos_table, const int* tokens, int vocab, int width, int pos0, int n_pos,
                                       const float* w, const float* b, float alpha) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= width) return;
    const int tok = tokens[t];
    const long long p = pos0 + t;
    float e = 0.0f, pv = 0.0f;
    if (tok >= 0 && tok < vocab) {
        if constexpr (sizeof(TT) == 2) e = __uint_as_float((uint32_t)table[(long long)tok * width + i] << 16); else e = table[(long long)tok * width + i];
    }
    if (p < n_pos) {
        if constexpr (sizeof(TT) == 2) pv = __uint_as_float((uint32_t)pos_table[p * width + i] << 16); else pv = pos_table[p * width + i];
    }
    float v = e + pv;
    if (w) v = fmaf(tanhf(alpha * v), w[i], b ? b[i] : 0.0f);
    out[t * width + i] = v;
    if (copy) copy[t * width + i] = v;
}

__global__ void sigmoid_gate_scaled_kernel(float* y, int ldy, const float* g, int ldg, const float* gb, float scale, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[t * ldy + i] = y[t * ldy + i] * sigmoidf_(g[t * ldg + i] + (gb ? gb[i] : 0.0f)) * scale;
}

__global__ void tanh_rows_kernel(float* x, int ldx, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[t * ldx + i] = tanhf(x[t * ldx + i]);
}

// one wave per (token, head): the head's dv values in registers (dv <= 64 * 16), mean of squares over the wave, weight, gate
constexpr int HRN_MAXC = 16;
__global__ __launch_bounds__(64) void head_rmsnorm_gate_kernel(float* y, int ldy, const float* x, int ldx, const float* w, int w_head_stride, const float* g, int ldg,
                                                               int act, float scale, int H, int dv, float eps) {
    const int lane = threadIdx.x, h = blockIdx.x % H;
    const long long t = blockIdx.x / H;
    const float* xr = x + t * ldx + (long long)h * dv;
    float v[HRN_MAXC];
    float ss = 0.0f;
#pragma unroll
    for (int c = 0; c < HRN_MAXC; ++c) {
        v[c] = c * 64 + lane < dv ? xr[c * 64 + lane] : 0.0f;
        ss = fmaf(v[c], v[c], ss);
    }
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
    for (int c = 0; c < HRN_MAXC; ++c) {
        const int i = c * 64 + lane;
        if (i >= dv) continue;
        float r = v[c] * inv * w[(long long)h * w_head_stride + i];
        if (act) {
            const float gg = g[t * ldg + (long long)h * dv + i];
            r *= act == 1 ? sigmoidf_(gg) : gg * sigmoidf_(gg);
        }
        y[t * ldy + (long long)h * dv + i] = r * scale;
    }
}

// The two gates in front of a mixer's output product, results as the bfloat16 rows that it reads (it would round them in a launch of its own: its image is read back in the next one).
// A lane has four entries on 16 bytes; LANES lanes share a head, the mean over its entries within them (entries beyond the head count as zero).  Bound by their bytes, of which the F32
// results, written and read again, were half.  us with the launch that rounded: 1999 rows of 16 heads of 128, norm and gate 18.9 + 8.6, now 11.2; 1024 rows of 2048, gate 6.2 + 5.1, now 5.3.
template <int LANES>
__global__ __launch_bounds__(256) void head_norm_gate_rows_kernel(uint16_t* y, const float* x, int ldx, const float* w, int w_head_stride, const float* g, int ldg, int act, float scale,
                                                                  long long heads, int H, int dv, float eps) {
    const long long at = blockIdx.x * (256LL / LANES) + threadIdx.x / LANES;
    if (at >= heads) return;                          // (whole groups of lanes)
    const int i = 4 * (threadIdx.x % LANES), h = (int)(at % H);
    const long long t = at / H;
    const bool in = i < dv;
    const float4 zero{0.0f, 0.0f, 0.0f, 0.0f};
    const float4 v = in ? load4(x + t * ldx + (long long)h * dv + i) : zero;
    const float4 wv = in ? load4(w + (long long)h * w_head_stride + i) : zero;
    const float4 gv = in && act ? load4(g + t * ldg + (long long)h * dv + i) : zero;
    float ss = square4(v, 0.0f);
#pragma unroll
    for (int m = LANES / 2; m; m >>= 1) ss += __shfl_xor(ss, m);
    const float inv = 1.0f / sqrtf(ss / (float)dv + eps);
    auto one = [&](float a, float b, float c) {
        float r = a * inv * b;
        if (act) r *= act == 1 ? sigmoidf_(c) : c * sigmoidf_(c);
        return r * scale;
    };
    if (in) *reinterpret_cast<uint2*>(y + at * dv + i) = pack4_bf16(float4{one(v.x, wv.x, gv.x), one(v.y, wv.y, gv.y), one(v.z, wv.z, gv.z), one(v.w, wv.w, gv.w)});
}

// per_head: entries that share a gate (0: a gate an entry)
__global__ __launch_bounds__(256) void gate_rows_kernel(uint16_t* y, const float* x, int ldx, const float* g, int ldg, int per_head, int n) {
    const long long t = blockIdx.y;
    const int i = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= n) return;
    const float4 v = load4(x + t * ldx + i);
    float4 c;
    if (per_head) { c.x = sigmoidf_(g[t * ldg + i / per_head]); c.y = c.z = c.w = c.x; }
    else {
        const float4 z = load4(g + t * ldg + i);
        c = float4{sigmoidf_(z.x), sigmoidf_(z.y), sigmoidf_(z.z), sigmoidf_(z.w)};
    }
    *reinterpret_cast<uint2*>(y + t * n + i) = pack4_bf16(float4{v.x * c.x, v.y * c.y, v.z * c.z, v.w * c.w});
}

struct SeamArgs {
    float* x; int ldx;
    const float* y; int ldy; const float* yb;
    const float* g; int ldg; const float* gb;
    float* hist; long long hist_stride; int n_hist; const float* coef;
    float* h; int ldh; const float* nw; const float* nb; float alpha;
    int n;
};
__global__ void gated_seam_kernel(const SeamArgs a) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    float r = a.x[t * a.ldx + i];
    if (a.y) {
        const float yy = a.y[t * a.ldy + i] + (a.yb ? a.yb[i] : 0.0f);
        r = fmaf(yy, sigmoidf_(a.g[t * a.ldg + i] + (a.gb ? a.gb[i] : 0.0f)), r);
    }
    if (a.n_hist > 0) {
        float s = 0.0f;
        for (int j = 0; j + 1 < a.n_hist; ++j) s = fmaf(a.coef[j], a.hist[j * a.hist_stride + t * a.n + i], s);
        a.hist[(a.n_hist - 1) * a.hist_stride + t * a.n + i] = r;
        r = fmaf(a.coef[a.n_hist - 1], r, s);
    }
    a.x[t * a.ldx + i] = r;
    if (a.h) a.h[t * a.ldh + i] = fmaf(tanhf(a.alpha * r), a.nw[i], a.nb ? a.nb[i] : 0.0f);
}

}  // namespace ntk

int ntk_dyt(float* y, int ldy, const float* x, int ldx, const float* w, const float* b, float alpha, int T, int n, void* stream) {
    if (!y || !x || !w) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::dyt_kernel, dim3((n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), y, ldy, x, ldx, w, b, alpha, n);
    return last_launch_status();
}

int ntk_embed_positions(float* out, float* copy, const void* table, const void* pos_table, int tdtype, const int* tokens, int T, int vocab, int width, int pos0,
                        int n_pos, const float* w, const float* b, float alpha, void* stream) {
    if (!out || !table || !pos_table || !tokens) return NTK_E_NULL;
    if (tdtype != NTK_DT_BF16 && tdtype != NTK_DT_F32) return NTK_E_DTYPE;
    if (T < 0 || vocab <= 0 || width <= 0 || pos0 < 0 || n_pos < 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    const dim3 grid((width + 255) / 256, T);
    if (tdtype == NTK_DT_BF16)
        hipLaunchKernelGGL(ntk::embed_positions_kernel<uint16_t>, grid, dim3(256), 0, resolve_stream(stream), out, copy, (const uint16_t*)table, (const uint16_t*)pos_table,
                           tokens, vocab, width, pos0, n_pos, w, b, alpha);
    else
        hipLaunchKernelGGL(ntk::embed_positions_kernel<float>, grid, dim3(256), 0, resolve_stream(stream), out, copy, (const float*)table, (const float*)pos_table, tokens,
                           vocab, width, pos0, n_pos, w, b, alpha);
    return last_launch_status();
}

int ntk_sigmoid_gate_scaled(float* y, int ldy, const float* g, int ldg, const float* gb, float scale, int T, int n, void* stream) {
    if (!y || !g) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldg < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::sigmoid_gate_scaled_kernel, dim3((n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), y, ldy, g, ldg, gb, scale, n);
    return last_launch_status();
}

int ntk_tanh_rows(float* x, int ldx, int T, int n, void* stream) {
    if (!x) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::tanh_rows_kernel, dim3((n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), x, ldx, n);
    return last_launch_status();
}

int ntk_head_rmsnorm_gate(float* y, int ldy, const float* x, int ldx, const float* w, int w_head_stride, const float* g, int ldg, int act, float scale, int T, int H,
                          int dv, float eps, void* stream) {
    if (!y || !x || !w || (act && !g)) return NTK_E_NULL;
    if (T < 0 || H <= 0 || dv <= 0 || dv > 64 * ntk::HRN_MAXC || act < 0 || act > 2 || ldy < H * dv || ldx < H * dv || (act && ldg < H * dv)) return NTK_E_SHAPE;
    if (w_head_stride != 0 && w_head_stride != dv) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::head_rmsnorm_gate_kernel, dim3(T * H), dim3(64), 0, resolve_stream(stream), y, ldy, x, ldx, w, w_head_stride, g, ldg, act, scale, H, dv, eps);
    return last_launch_status();
}

// whole groups of four on 16 bytes, a head within a wave
namespace ntk {
static bool fours(int a, int b, int c, const void* p, const void* q) { return !((a | b | c) & 3) && !(((uintptr_t)p | (uintptr_t)q) & 15); }
}

int ntk_head_rmsnorm_gate_16(void* y16, const float* x, int ldx, const float* w, int w_head_stride, const float* g, int ldg, int act, float scale, int T, int H, int dv, float eps,
                             void* stream) {
    if (!y16 || !x || !w || (act && !g)) return NTK_E_NULL;
    if (T < 0 || H <= 0 || dv <= 0 || act < 0 || act > 2 || w_head_stride < 0 || ldx < H * dv || (act && ldg < H * dv)) return NTK_E_SHAPE;
    if (dv > 256 || !ntk::fours(dv, ldx, w_head_stride, x, w) || !ntk::fours(act ? ldg : 0, 0, 0, act ? g : nullptr, nullptr) || ((uintptr_t)y16 & 7)) return NTK_E_ALIGN;
    if (T == 0) return NTK_OK;
    const long long heads = (long long)T * H;
    auto launch = [&](auto kernel, int lanes) {
        const long long per = 256 / lanes;
        hipLaunchKernelGGL(kernel, dim3((unsigned)((heads + per - 1) / per)), dim3(256), 0, resolve_stream(stream), (uint16_t*)y16, x, ldx, w, w_head_stride, g, ldg, act, scale, heads, H, dv, eps);
    };
    if (dv <= 64) launch(ntk::head_norm_gate_rows_kernel<16>, 16);
    else if (dv <= 128) launch(ntk::head_norm_gate_rows_kernel<32>, 32);
    else launch(ntk::head_norm_gate_rows_kernel<64>, 64);
    return last_launch_status();
}

int ntk_gate_rows_16(void* y16, const float* x, int ldx, const float* g, int ldg, int per_head, int T, int n, void* stream) {
    if (!y16 || !x || !g) return NTK_E_NULL;
    if (T < 0 || T > 65535 || n <= 0 || per_head < 0 || (per_head && n % per_head) || ldx < n || ldg < (per_head ? n / per_head : n)) return NTK_E_SHAPE;
    if (!ntk::fours(n, ldx, per_head ? per_head : ldg, x, per_head ? nullptr : g) || ((uintptr_t)y16 & 7)) return NTK_E_ALIGN;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::gate_rows_kernel, dim3((n / 4 + 255) / 256, T), dim3(256), 0, resolve_stream(stream), (uint16_t*)y16, x, ldx, g, ldg, per_head, n);
    return last_launch_status();
}

int ntk_gated_seam(const ntk_gated_seam_desc* d, void* stream) {
    if (!d || !d->x || (d->y && !d->g) || (d->n_hist > 0 && (!d->hist || !d->coef)) || (d->h && !d->nw)) return NTK_E_NULL;
    if (d->T < 0 || d->n <= 0 || d->ldx < d->n || (d->y && (d->ldy < d->n || d->ldg < d->n)) || (d->h && d->ldh < d->n) || d->n_hist < 0) return NTK_E_SHAPE;
    if (d->n_hist > 0 && d->hist_stride < (long long)d->T * d->n) return NTK_E_SHAPE;
    if (d->T == 0) return NTK_OK;
    ntk::SeamArgs a{d->x, d->ldx, d->y, d->ldy, d->yb, d->g, d->ldg, d->gb, d->hist, d->hist_stride, d->n_hist, d->coef, d->h, d->ldh, d->nw, d->nb, d->alpha, d->n};
    hipLaunchKernelGGL(ntk::gated_seam_kernel, dim3((d->n + 255) / 256, d->T), dim3(256), 0, resolve_stream(stream), a);
    return last_launch_status();
}

// ---------------------------------------------------------------------------------------------------------------- layers with scaled, RMS-normed sublayer results
// The seam between two sublayers: the result the stream is still owed joins it (RMS norm, weight, a fixed factor), and the norm in front of the next sublayer
// reads the row the same launch has just written (a thread reads back only what it wrote itself).  The short convolution of a recurrent mixer's projections
// carries its last inputs from portion to portion; one token is one launch (a channel's history belongs to the thread that owns the channel).
namespace ntk {

template <int NT>
__global__ __launch_bounds__(NT) void rms_seam_kernel(float* h, int ldh, float* x, int ldx, const float* add_y, int ldy, const float* add_w, float mult, const float* w,
                                                      int n, float eps) {
    __shared__ float red[16];
    constexpr int KEEP = 4096 / NT;              // a thread's first entries stay in registers: rows up to 4096 wide cross memory once
    float* xr = x + (long long)blockIdx.x * ldx;
    float v[KEEP];
    if (add_y) {
        const float* yr = add_y + (long long)blockIdx.x * ldy;
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < KEEP; ++k) {
            const int i = threadIdx.x + NT * k;
            v[k] = i < n ? yr[i] : 0.0f;
            ss = fmaf(v[k], v[k], ss);
        }
        for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) ss = fmaf(yr[i], yr[i], ss);
        const float inv = mult / sqrtf(block_sum(ss, red) / (float)n + eps);
#pragma unroll
        for (int k = 0; k < KEEP; ++k) {
            const int i = threadIdx.x + NT * k;
            if (i < n) { v[k] = fmaf(v[k] * inv, add_w[i], xr[i]); xr[i] = v[k]; }
        }
        for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) xr[i] = fmaf(yr[i] * inv, add_w[i], xr[i]);
    } else {
#pragma unroll
        for (int k = 0; k < KEEP; ++k) {
            const int i = threadIdx.x + NT * k;
            v[k] = i < n ? xr[i] : 0.0f;
        }
    }
    if (!h) return;                              // (uniform over the launch)
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < KEEP; ++k)
        if ((int)threadIdx.x + NT * k < n) ss = fmaf(v[k], v[k], ss);
    for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) ss = fmaf(xr[i], xr[i], ss);
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + eps);
    float* hr = h + (long long)blockIdx.x * ldh;
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
        const int i = threadIdx.x + NT * k;
        if (i < n) hr[i] = v[k] * inv * w[i];
    }
    for (int i = threadIdx.x + NT * KEEP; i < n; i += NT) hr[i] = xr[i] * inv * w[i];
}

constexpr int kConvMaxTaps = 16;
__device__ __forceinline__ float conv_act(float s, int act) { return act == 1 ? s / (1.0f + expf(-s)) : s; }

// the input `back` rows before row t of the portion: the portion's own row, a carried one, or zero before the sequence's start
__device__ __forceinline__ float conv_input(const float* x, int ldx, const float* state, int taps, int pos0, int n, int c, int idx) {
    if (idx >= 0) return x[(long long)idx * ldx + c];
    if (pos0 + idx < 0) return 0.0f;
    return state[(long long)(taps - 1 + idx) * n + c];   // carried row taps - 1 + idx: the row that lay idx before this portion
}

// Up to four taps, channels in fours on 16 bytes: a thread owns four channels of eight rows, reads a row once for all the outputs that take it, and the first tile's threads, the
// only ones that read the carried rows, leave the new ones behind: one launch.  Bound by its bytes; 4096 channels of 1024 rows: 14.8 us, an output a thread and the
// carried rows in a launch of their own 22.8 + 4.7.
constexpr int kConvRows = 8, kConvRowTaps = 4;
__global__ __launch_bounds__(256) void causal_conv_rows_kernel(float* y, int ldy, const float* x, int ldx, const float* w, float* state, int taps, int act, int pos0, int T, int n) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, t0 = blockIdx.y * kConvRows, skip = kConvRowTaps - taps;
    if (c >= n) return;
    auto input = [&](int idx) -> f4 {                         // (conv_input's rule)
        if (idx >= 0) return *reinterpret_cast<const f4*>(x + (long long)idx * ldx + c);
        if (pos0 + idx < 0) return f4{0.0f, 0.0f, 0.0f, 0.0f};
        return *reinterpret_cast<const f4*>(state + (long long)(taps - 1 + idx) * n + c);
    };
    f4 in[kConvRows + kConvRowTaps - 1], ws[kConvRowTaps];
#pragma unroll
    for (int i = 0; i < kConvRows + kConvRowTaps - 1; ++i)
        if (i >= skip) in[i] = input(min(t0 - (kConvRowTaps - 1) + i, T - 1));
#pragma unroll
    for (int j = 0; j < kConvRowTaps; ++j)
        if (j >= skip)
#pragma unroll
            for (int e = 0; e < 4; ++e) ws[j][e] = w[(long long)(c + e) * taps + j - skip];
#pragma unroll
    for (int r = 0; r < kConvRows; ++r) {
        if (t0 + r >= T) break;
        f4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < kConvRowTaps; ++j)
            if (j >= skip)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = fmaf(ws[j][e], in[r + j][e], s[e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = conv_act(s[e], act);
        *reinterpret_cast<f4*>(y + (long long)(t0 + r) * ldy + c) = s;
    }
    if (blockIdx.y || taps == 1) return;
    f4 keep[kConvRowTaps - 1];
#pragma unroll
    for (int r = 1; r < kConvRowTaps; ++r)
        if (r < taps) keep[r - 1] = input(T - taps + r);
#pragma unroll
    for (int r = 1; r < kConvRowTaps; ++r)
        if (r < taps) *reinterpret_cast<f4*>(state + (long long)(r - 1) * n + c) = keep[r - 1];
}

// blocks y < T: the outputs; one more launch shifts the carried rows (they are read here)
__global__ void causal_conv_act_kernel(float* y, int ldy, const float* x, int ldx, const float* w, const float* state, int taps, int act, int pos0, int n) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (c >= n) return;
    float s = 0.0f;
    for (int j = 0; j < taps; ++j) s = fmaf(w[(long long)c * taps + j], conv_input(x, ldx, state, taps, pos0, n, c, t - (taps - 1) + j), s);
    y[(long long)t * ldy + c] = conv_act(s, act);
}

// the carried rows after the portion: a thread owns a channel, reads its taps - 1 new rows (some of them old carried rows when the portion is shorter) and
// then writes them.  T == 1 with an output: the whole operator for one token in this one launch.
__global__ void causal_conv_carry_kernel(float* y, const float* x, int ldx, const float* w, float* state, int taps, int act, int pos0, int T, int n) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    float keep[kConvMaxTaps];
#pragma unroll
    for (int r = 0; r < kConvMaxTaps; ++r)
        if (r < taps) keep[r] = conv_input(x, ldx, state, taps, pos0, n, c, T - taps + r);      // rows T - taps .. T - 1 (the first only for the output)
    if (y) {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < kConvMaxTaps; ++r)
            if (r < taps) s = fmaf(w[(long long)c * taps + r], keep[r], s);
        y[c] = conv_act(s, act);
    }
#pragma unroll
    for (int r = 1; r < kConvMaxTaps; ++r)
        if (r < taps) state[(long long)(r - 1) * n + c] = keep[r];
}

__global__ void softcap_rows_kernel(float* x, int ldx, float cap, int n) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[t * ldx + i] = cap * tanhf(x[t * ldx + i] / cap);
}

__global__ void head_gate_kernel(float* y, int ldy, const float* g, int ldg, int H, int dv) {
    const long long t = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= H * dv) return;
    y[t * ldy + i] *= sigmoidf_(g[t * ldg + i / dv]);
}

}  // namespace ntk

int ntk_rms_seam(float* h, int ldh, float* x, int ldx, const float* add_y, int ldy, const float* add_w, float mult, const float* w, int T, int n, float eps,
                 void* stream) {
    if (!x || (add_y && !add_w) || (h && !w)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n || (h && ldh < n) || (add_y && ldy < n)) return NTK_E_SHAPE;
    if (T == 0 || (!add_y && !h)) return NTK_OK;
    if (T <= kFewRows) hipLaunchKernelGGL(ntk::rms_seam_kernel<1024>, dim3(T), dim3(1024), 0, resolve_stream(stream), h, ldh, x, ldx, add_y, ldy, add_w, mult, w, n, eps);
    else hipLaunchKernelGGL(ntk::rms_seam_kernel<256>, dim3(T), dim3(256), 0, resolve_stream(stream), h, ldh, x, ldx, add_y, ldy, add_w, mult, w, n, eps);
    return last_launch_status();
}

int ntk_rms_seam_16(void* h16, float* x, int ldx, const float* add_y, int ldy, const float* add_w, float mult, const float* w, int T, int n, float eps, void* stream) {
    if (!h16 || !x || !w || (add_y && !add_w)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n || (add_y && ldy < n)) return NTK_E_SHAPE;
    if (!whole_rows(n, ldx, add_y ? ldy : 0, x, add_y, w) || !whole_rows(n, 0, 0, add_y ? add_w : nullptr, nullptr, nullptr) || ((uintptr_t)h16 & 7)) return NTK_E_ALIGN;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::rows_seam_kernel, dim3(T), dim3(256), 0, resolve_stream(stream), (uint16_t*)h16, x, ldx, add_y, ldy, add_w, mult, w, n, eps);
    return last_launch_status();
}

int ntk_causal_conv_act(float* y, int ldy, const float* x, int ldx, const float* w, float* state, int taps, int act, int pos0, int T, int n, void* stream) {
    if (!y || !x || !w || (taps > 1 && !state)) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldy < n || ldx < n || taps < 1 || taps > ntk::kConvMaxTaps || pos0 < 0 || act < 0 || act > 1) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipStream_t s = resolve_stream(stream);
    if (T == 1) {
        hipLaunchKernelGGL(ntk::causal_conv_carry_kernel, dim3((n + 255) / 256), dim3(256), 0, s, y, x, ldx, w, state, taps, act, pos0, T, n);
        return last_launch_status();
    }
    const uintptr_t at = (uintptr_t)y | (uintptr_t)x | (uintptr_t)(taps > 1 ? state : nullptr);
    // (a thread of the rows' form walks eight rows: with less than about a million results there are too few of them.  us, both launches of the other form and this one: 4096 channels, 40
    // rows 5.1 and 8.0, 200 8.0 and 8.3, 400 11.7 and 9.0; 1024 channels, 400 rows 6.2 and 8.0, 1000 8.9 and 8.3; 12288 channels, 64 rows 7.9 and 8.4, 100 9.8 and 8.6)
    if (taps <= ntk::kConvRowTaps && (long long)T * n >= 7 << 17 && !((n | ldx | ldy) & 3) && !(at & 15)) {
        hipLaunchKernelGGL(ntk::causal_conv_rows_kernel, dim3((n / 4 + 255) / 256, (T + ntk::kConvRows - 1) / ntk::kConvRows), dim3(256), 0, s, y, ldy, x, ldx, w, state, taps, act, pos0, T, n);
        return last_launch_status();
    }
    hipLaunchKernelGGL(ntk::causal_conv_act_kernel, dim3((n + 255) / 256, T), dim3(256), 0, s, y, ldy, x, ldx, w, (const float*)state, taps, act, pos0, n);
    const int st = last_launch_status();
    if (st != NTK_OK || taps == 1) return st;
    hipLaunchKernelGGL(ntk::causal_conv_carry_kernel, dim3((n + 255) / 256), dim3(256), 0, s, (float*)nullptr, x, ldx, w, state, taps, act, pos0, T, n);
    return last_launch_status();
}

int ntk_softcap_rows(float* x, int ldx, float cap, int T, int n, void* stream) {
    if (!x) return NTK_E_NULL;
    if (T < 0 || n <= 0 || ldx < n || !(cap > 0.0f)) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::softcap_rows_kernel, dim3((n + 255) / 256, T), dim3(256), 0, resolve_stream(stream), x, ldx, cap, n);
    return last_launch_status();
}

int ntk_head_gate(float* y, int ldy, const float* g, int ldg, int T, int H, int dv, void* stream) {
    if (!y || !g) return NTK_E_NULL;
    if (T < 0 || H <= 0 || dv <= 0 || ldy < H * dv || ldg < H) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    hipLaunchKernelGGL(ntk::head_gate_kernel, dim3((H * dv + 255) / 256, T), dim3(256), 0, resolve_stream(stream), y, ldy, g, ldg, H, dv);
    return last_launch_status();
}
