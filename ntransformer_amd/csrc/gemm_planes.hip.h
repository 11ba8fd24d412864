// gemm_planes.hip.h -- the FP16 GEMM's operand planes: their layout in its workspace, and the split that leaves a short prompt's planes from the launch that produces its values
// (gemm_f16.hip: the GEMM and most producers; attention_mfma.hip: a short prompt's attention).
#pragma once
#include "common.hip.h"

namespace ntk {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int GB_TOK = 64;           // tokens per pass
constexpr int GB_MAX_CHUNKS = 16;   // 64-token chunks per launch (32 measured no better: 15.1k vs 16.0k tok/s at 2048 tokens)
constexpr int GB_PIECE = 1024;       // bytes of one (step, plane, token block) operand record
constexpr int GB_PLANES = 2;         // FP16 pieces of an activation
constexpr int GB_STEP_BYTES = GB_PLANES * 4 * GB_PIECE;   // 8 KB of activation operands per step
constexpr int GB_AUX_BYTES = GB_TOK * 4;                  // per step: one eighth of its unit's record of sums (K-quant minimum term)
constexpr int GB_SHORT = 32;         // tokens of a short prompt (gemm_quant_f16_kslice_kernel), whose planes are scaled per GB_GROUP columns
constexpr int GB_GROUP = 256;
constexpr int GB_MIN_UNIT_BYTES = 8 * GB_AUX_BYTES;       // per unit of 8 steps and 64-token chunk: 2 pieces x 4 token blocks x 2 x 16 tokens x 4 steps x FP16

// exponent field of s from the token's largest |x| (bit pattern; a NaN pattern counts as the largest binade: any scale will do then)
__device__ __forceinline__ int scale_exp_of_max(uint32_t max_bits) {
    const int em = (int)((max_bits >> 23) & 0xFFu);
    return min(253, max(1, 268 - em));
}
// Layout of the workspace: [chunk][(in / 32 + 1) step records of 8 KB | sums of the units], then [1 / s][s] of the pass
static __host__ __device__ size_t ws_chunk_bytes(int in) {
    return ((size_t)(in / 32 + 1) * GB_STEP_BYTES + (size_t)((in / 32 + 15) / 8) * GB_MIN_UNIT_BYTES + 255) / 256 * 256;
}
constexpr size_t GB_SCALE_BYTES = 2 * GB_MAX_CHUNKS * GB_TOK * sizeof(float);   // the launch's 1 / s and s
// ... and, in the second chunk's area (a short prompt has one chunk), for the short prompts' form: [GB_GROUP columns][GB_SHORT tokens] 1 / s, then [512 columns][GB_SHORT tokens] sums of squares (short_split below)
static __host__ __device__ size_t ws_group_floats(int in) { return (size_t)((in + GB_GROUP - 1) / GB_GROUP) * GB_SHORT; }
static __host__ __device__ size_t ws_group_offset(int in) { return ws_chunk_bytes(in); }   // (fits: a 128th of the chunk's records at most)
static __host__ __device__ size_t ws_part_offset(int in) { return (size_t)GB_MAX_CHUNKS * ws_chunk_bytes(in) + GB_SCALE_BYTES; }
// Half a wave splits a token's group of columns: lane l of its 32 holds in x[8] the values of columns 32 step + 4 g + {0 .. 3, 16 .. 19}, step = the group's first + l / 4, g = l % 4; steps
// past the row hold zeros.  t: the token, < 0: nothing is written.
__device__ __forceinline__ void short_split(float (&x)[8], int step, int g, int t, int in, uint8_t* __restrict__ ws) {
    uint32_t mb = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) mb = max(mb, __float_as_uint(x[e]) & 0x7FFFFFFFu);   // (bit patterns: ordered like the values, and a NaN is not dropped)
#pragma unroll
    for (int o = 1; o <= 16; o <<= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
    const int es = scale_exp_of_max(mb);
    const float sc = __uint_as_float((uint32_t)es << 23);
    float p1[8], p2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        x[e] *= sc;
        const _Float16 h1 = (_Float16)x[e];
        p1[e] = (float)h1;
        p2[e] = x[e] - p1[e];
    }
    auto pk = [](float lo, float hi) {
        const f16x2 h = {(_Float16)lo, (_Float16)hi};
        return __builtin_bit_cast(uint32_t, h);
    };
    float sum = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (t < 0 || step * 32 >= in) return;
    const int tb = t >> 4, j = t & 15;
    u32x4* xb = reinterpret_cast<u32x4*>(ws);
    const size_t base = ((size_t)step * GB_PLANES * 4 + tb) * 64 + (j + 16 * g);
    xb[base] = u32x4{pk(p1[0], p1[1]), pk(p1[2], p1[3]), pk(p1[4], p1[5]), pk(p1[6], p1[7])};
    xb[base + 256] = u32x4{pk(p2[0], p2[1]), pk(p2[2], p2[3]), pk(p2[4], p2[5]), pk(p2[6], p2[7])};
    if (g == 0) {
        const float y = sum * 0.015625f;
        const _Float16 h1 = (_Float16)y, h2 = (_Float16)(y - (float)h1);
        _Float16* rec = reinterpret_cast<_Float16*>(ws + (size_t)(in / 32 + 1) * GB_STEP_BYTES + (size_t)(step >> 3) * GB_MIN_UNIT_BYTES);
        const int pos = ((tb * 2 + ((step >> 2) & 1)) * 64 + j * 4 + (step & 3));
        rec[pos] = h1;
        rec[4 * 128 + pos] = h2;
        if (step % (GB_GROUP / 32) == 0) reinterpret_cast<float*>(ws + ws_group_offset(in))[step / (GB_GROUP / 32) * GB_SHORT + t] = __uint_as_float((uint32_t)(254 - es) << 23);
    }
}

}  // namespace ntk
