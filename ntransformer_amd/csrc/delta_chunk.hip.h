// delta_chunk.hip.h -- the delta rule with one gate per head, 32 tokens at a time on the matrix instructions.  Included by gated_recurrence.hip.
//
//     S_t = w_t S_(t-1) + u_t d_t^T,   d_t = a_t v_t - a_t w_t S_(t-1)^T u_t,   o_t = S_t^T q_t                    (u_t: the unit key, q_t: scaled)
//
// With W_t = w_1 ... w_t inside a chunk and R[t][s] = w_(s+1) ... w_t (running products of the decays: nothing is divided by one, whatever they are), the chunk's
// d follow from the state S_0 at its start by a unit lower triangular system:
//
//     (I + A) D = diag(a) V - diag(a W) U S_0,   A[t][s] = a_t R[t][s] (u_t . u_s), s < t
//     o_t = W_t S_0^T q_t + sum_(s <= t) R[t][s] (q_t . u_s) d_s,   S_C = W_C S_0 + sum_s R[C][s] u_s d_s^T
//
// Everything that does not know S_0 is one launch over all chunks and heads at once (delta_chunk_solve_kernel: unit vectors and gates from the raw projections, the two
// 32 x 32 products, forward substitution on [diag(a) V | diag(a W) U] with a thread per column); what is left from chunk to chunk is four small products per head
// and 16 value columns (delta_chunk_walk_kernel), the state in the accumulators of its waves all the way.  1024 tokens of 16 heads of 128 x 128: 74 us, where the walk
// token by token, its pre-pass and the settling of its segments took 277.
//
// The products that the walk waits for take every F32 value as three bfloat16 pieces (8 + 8 + 8 bits: nothing of the value is lost, its exponent's range is F32's own) and
// six products of pieces, all but those below 2^-25 of the value: K = 32 in 6 x 16 cycles where the F32 instruction takes 8 x 32.  The solve leaves its results as pieces in
// the order of the operand slots; the state and the chunk's d are taken apart on their way through LDS.
#pragma once

namespace ntk {

constexpr int kDeltaChunk = 32;
typedef float deltax4_t __attribute__((ext_vector_type(4)));
typedef uint32_t deltap_t __attribute__((ext_vector_type(4)));

struct DeltaArgs {
    RecArgs r;
    int chunks;
    float *vt;                             // per (chunk, head): [dv][32]
    deltap_t *ut, *qw, *udt, *pm;          // operand slots [piece][lane] of 8 x bfloat16: per (chunk, head) and [token half][32 channels], the same, [16 channels], [token half]
    float* wc;                             // one number
};

// the element of an operand slot: lane (m = lane % 16, g = lane / 16) holds row (column) m at the eight places 4 g + {0 .. 3} and 16 + 4 g + {0 .. 3} of a step of 32 -- the
// accumulators of two waves (rows 4 g + r of 16 each) are then a slot as they stand
__device__ __forceinline__ int delta_place(int g, int j) { return 4 * g + (j & 3) + 16 * (j >> 2); }

// four values -> three pieces of two dwords each.  (Not finite: the first piece holds it, the others are zero.  Above the largest bfloat16: that, not the infinity it would round to.)
struct DeltaPieces { uint32_t w[3][2]; };
__device__ __forceinline__ DeltaPieces delta_split(deltax4_t x) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    constexpr float top = 3.3895314e38f;
    DeltaPieces p;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float a = x[2 * h], b = x[2 * h + 1];
        const bool fa = fabsf(a) < INFINITY, fb = fabsf(b) < INFINITY;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(i == 0 ? f2{fa ? __builtin_amdgcn_fmed3f(a, -top, top) : a, fb ? __builtin_amdgcn_fmed3f(b, -top, top) : b} : f2{a, b}, b2));
            p.w[i][h] = w;
            a = fa ? a - __uint_as_float(w << 16) : 0.0f;
            b = fb ? b - __uint_as_float(w & 0xFFFF0000u) : 0.0f;
        }
    }
    return p;
}
__device__ __forceinline__ void delta_put(deltap_t* slot, deltax4_t lo, deltax4_t hi) {
    const DeltaPieces a = delta_split(lo), b = delta_split(hi);
#pragma unroll
    for (int i = 0; i < 3; ++i) slot[64 * i] = deltap_t{a.w[i][0], a.w[i][1], b.w[i][0], b.w[i][1]};
}
// small += the five products of pieces that correct the first, large += the first
__device__ __forceinline__ void delta_mul(deltax4_t& large, deltax4_t& small, const deltap_t (&x)[3], const deltap_t (&y)[3]) {
    typedef __bf16 b8 __attribute__((ext_vector_type(8)));
    auto op = [](const deltap_t& v) { return __builtin_bit_cast(b8, v); };
    small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[2]), op(y[0]), small, 0, 0, 0);
    large = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[0]), op(y[0]), large, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[0]), op(y[2]), small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[1]), op(y[1]), small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[1]), op(y[0]), small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op(x[0]), op(y[1]), small, 0, 0, 0);
}

// floats of DeltaArgs' buffers
inline size_t delta_chunk_floats(int T, int H, int dn, int dv) {
    const size_t blocks = (size_t)((T + kDeltaChunk - 1) / kDeltaChunk) * H;
    return blocks * ((size_t)kDeltaChunk * (dv + (3 * dn + kDeltaChunk) / 2 * 3) + 4);   // (a piece is half a float, three to a value)
}

// grid (chunks, H).  A chain of short steps (loads, norms, products, substitution) on a launch of one or two workgroups a CU, so every instruction is fetched cold: the
// code stays small.  The substitution goes four rows at a time in a loop, the solved rows of a thread's column in LDS; unrolled over all 32 rows with the column in
// registers it was 20 KB of straight-line code, and 47 us at 32 chunks of 16 heads (24 us at 5) against 21 (16).
template <int DN>
__global__ __launch_bounds__(256) void delta_chunk_solve_kernel(const DeltaArgs A) {
    constexpr int C = kDeltaChunk, LD = DN + 4, LA = C + 4;
    __shared__ __attribute__((aligned(16))) float us[C * LD], qs[C * LD], am[C * LA], xs[C][256];
    __shared__ float rm[C][C + 1], wv[C], av[C], cw[C];
    const RecArgs& a = A.r;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.y;
    const int t0 = blockIdx.x * C, nt = min(C, a.T - t0);
    const long long blk = (long long)blockIdx.x * a.H + h;
    {   // eight lanes a token: unit vectors; rows past the end: a token that changes nothing
        const int row = tid / 8, sub = tid % 8;
        const bool ok = row < nt;
        const long long t = t0 + min(row, nt - 1), oq = (long long)(a.G > 0 ? h / (a.H / a.G) : h) * a.dn;
        float4 k4[DN / 32], q4[DN / 32];
#pragma unroll
        for (int i = 0; i < DN / 32; ++i) {
            k4[i] = *reinterpret_cast<const float4*>(a.k + t * a.ldk + oq + 32 * i + 4 * sub);
            q4[i] = *reinterpret_cast<const float4*>(a.q + t * a.ldq + oq + 32 * i + 4 * sub);
        }
        const float z = a.wz[t * a.ldw + h] + (a.wb ? a.wb[h] : 0.0f), y = a.az[t * a.lda + h] + (a.ab ? a.ab[h] : 0.0f);
        float ss = 0.0f, sq = 0.0f;
#pragma unroll
        for (int i = 0; i < DN / 32; ++i) {
            ss = fmaf(k4[i].x, k4[i].x, ss); ss = fmaf(k4[i].y, k4[i].y, ss); ss = fmaf(k4[i].z, k4[i].z, ss); ss = fmaf(k4[i].w, k4[i].w, ss);
            sq = fmaf(q4[i].x, q4[i].x, sq); sq = fmaf(q4[i].y, q4[i].y, sq); sq = fmaf(q4[i].z, q4[i].z, sq); sq = fmaf(q4[i].w, q4[i].w, sq);
        }
        const float km = 1.0f / sqrtf(group_sum<8>(ss) + a.unit_eps);
        const float qsum = group_sum<8>(sq), qm = a.unit_q ? a.q_scale / sqrtf(qsum + a.unit_eps) : a.q_scale;
#pragma unroll
        for (int i = 0; i < DN / 32; ++i) {
            const float4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            *reinterpret_cast<float4*>(us + row * LD + 32 * i + 4 * sub) = ok ? float4{k4[i].x * km, k4[i].y * km, k4[i].z * km, k4[i].w * km} : zero;
            *reinterpret_cast<float4*>(qs + row * LD + 32 * i + 4 * sub) = ok ? float4{q4[i].x * qm, q4[i].y * qm, q4[i].z * qm, q4[i].w * qm} : zero;
        }
        if (sub == 0) {
            wv[row] = ok ? decay_of(z, a.decay_form, a.decay_rates ? a.decay_rates[h] : a.decay_param) : 1.0f;
            av[row] = ok ? 1.0f / (1.0f + expf(-y)) : 0.0f;
        }
    }
    __syncthreads();
    if (tid < C) {                                            // R[.][tid], down the column
        float p = 1.0f;
#pragma unroll
        for (int t = 0; t < C; ++t) {
            if (t > tid) p *= wv[t];
            rm[t][tid] = p;
        }
    } else if (tid == C) {
        float p = 1.0f;
#pragma unroll
        for (int t = 0; t < C; ++t) { p *= wv[t]; cw[t] = p; }
        A.wc[blk] = p;
    }
    // the 16 x 16 tiles on and below the diagonal of U U^T and Q U^T
    const int m = lane & 15, g = lane >> 4;
    deltax4_t acc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tile = wave + 4 * u, ti = tile % 3 > 0, tj = tile % 3 == 2;
        acc[u] = deltax4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (tile >= 6) break;
        const float* x = (tile < 3 ? us : qs) + (16 * ti + m) * LD + 4 * g;
        const float* y = us + (16 * tj + m) * LD + 4 * g;
#pragma unroll 2
        for (int k = 0; k < DN; k += 16) {
            const float4 x4 = *reinterpret_cast<const float4*>(x + k), y4 = *reinterpret_cast<const float4*>(y + k);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x4.x, y4.x, acc[u], 0, 0, 0);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x4.y, y4.y, acc[u], 0, 0, 0);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x4.z, y4.z, acc[u], 0, 0, 0);
            acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(x4.w, y4.w, acc[u], 0, 0, 0);
        }
    }
    __syncthreads();
    float* pm = &xs[0][0];                                    // [32][LA], until the substitution takes the room
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tile = wave + 4 * u, ti = tile % 3 > 0, tj = tile % 3 == 2, s = 16 * tj + m;
        if (tile >= 6) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * ti + 4 * g + r;
            if (tile < 3) am[t * LA + s] = s < t ? av[t] * rm[t][s] * acc[u][r] : 0.0f;
            else pm[t * LA + s] = s <= t ? rm[t][s] * acc[u][r] : 0.0f;
        }
    }
    pm[(tid / 16) * LA + 16 + tid % 16] = 0.0f;                // the tile above the diagonal (256 threads: 16 x 16)
    __syncthreads();
    // W q, the keys with what decays behind them, and the products of queries and keys, as operand slots
    constexpr int NS = DN / 32;
    const int pg = 4 * ((tid & 63) >> 4), pr = tid & 15;      // (a thread's slot has the same lane in every round)
#pragma unroll 2
    for (int e = tid; e < 2 * NS * 64; e += 256) {
        const int q = e / 64, t = 16 * (q / NS) + pr;
        const float* x = qs + t * LD + 32 * (q % NS) + pg;
        delta_put(A.qw + (blk * 2 * NS + q) * 192 + lane, cw[t] * *reinterpret_cast<const deltax4_t*>(x), cw[t] * *reinterpret_cast<const deltax4_t*>(x + 16));
    }
#pragma unroll 2
    for (int e = tid; e < DN / 16 * 64; e += 256) {
        const float *u = us + pg * LD + 16 * (e / 64) + pr, *w = rm[C - 1] + pg;
        delta_put(A.udt + (blk * (DN / 16) + e / 64) * 192 + lane, deltax4_t{w[0] * u[0], w[1] * u[LD], w[2] * u[2 * LD], w[3] * u[3 * LD]},
                  deltax4_t{w[16] * u[16 * LD], w[17] * u[17 * LD], w[18] * u[18 * LD], w[19] * u[19 * LD]});
    }
    if (tid < 128) {
        const float* x = pm + (16 * (tid / 64) + pr) * LA + pg;
        delta_put(A.pm + (blk * 2 + tid / 64) * 192 + lane, *reinterpret_cast<const deltax4_t*>(x), *reinterpret_cast<const deltax4_t*>(x + 16));
    }
    __syncthreads();                                          // (pm lies in xs)
    // forward substitution, a column a thread: the values', then the keys'
    for (int c = tid; c < a.dv + DN; c += 256) {
        const bool value = c < a.dv;
        const float* v = a.v + (long long)t0 * a.ldv + (long long)h * a.dv + c;
        auto right = [&](int t) -> float { return value ? (t < nt ? v[(long long)t * a.ldv] : 0.0f) : t < C ? cw[t] * us[t * LD + c - a.dv] : 0.0f; };
        float next[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) next[i] = right(i);
        for (int t = 0; t < C; t += 4) {
            float x[4], y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 4; ++i) { x[i] = next[i] * av[t + i]; next[i] = right(t + 4 + i); }
#pragma unroll 2
            for (int s = 0; s < t; s += 4) {
                float xv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) xv[j] = xs[s + j][tid];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 a4 = *reinterpret_cast<const float4*>(am + (t + i) * LA + s);
                    y[i] = fmaf(a4.x, xv[0], y[i]); y[i] = fmaf(a4.y, xv[1], y[i]); y[i] = fmaf(a4.z, xv[2], y[i]); y[i] = fmaf(a4.w, xv[3], y[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < i; ++j) y[i] = fmaf(am[(t + i) * LA + t + j], x[j], y[i]);
                x[i] -= y[i];
                xs[t + i][tid] = x[i];
            }
            if (value) *reinterpret_cast<float4*>(A.vt + (blk * a.dv + c) * C + t) = float4{x[0], x[1], x[2], x[3]};
            else
#pragma unroll
                for (int i = 0; i < 4; ++i) us[(t + i) * LD + c - a.dv] = x[i];   // (its own column, behind what it has read)
        }
    }
    __syncthreads();
#pragma unroll 2
    for (int e = tid; e < 2 * NS * 64; e += 256) {
        const float* x = us + (16 * (e / 64 / NS) + pr) * LD + 32 * (e / 64 % NS) + pg;
        delta_put(A.ut + (blk * 2 * NS + e / 64) * 192 + lane, *reinterpret_cast<const deltax4_t*>(x), *reinterpret_cast<const deltax4_t*>(x + 16));
    }
}

// grid (H, dv / 16) -- the column blocks of a head, which read the same operands, fall on the same L2 where H is a multiple of the eight --, a wave per 16 key channels.
// Wave w's accumulators are rows 16 w ... of the 16 columns.  Per chunk: every wave leaves its rows' pieces in LDS, the first four take a 16 x 16 tile of U' S_0 and W Q S_0
// each, D = V' - U' S_0 goes back through LDS, then the state's update everywhere and the outputs' product with D in two waves.  Bound by this chain of two barriers a
// chunk; operands are requested two chunks ahead.  1024 tokens of 16 heads of 128 x 128: 49 us (F32 instructions, every wave a share of all four tiles: 72).
template <int DN>
__global__ __launch_bounds__(4 * DN, DN / 64) void delta_chunk_walk_kernel(const DeltaArgs A) {
    constexpr int C = kDeltaChunk, NW = DN / 16, NS = DN / 32;
    static_assert(NW >= 4, "a wave per tile");
    __shared__ deltap_t sb[3][NS][64], db[3][64];
    const RecArgs& a = A.r;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const int h = blockIdx.x, c0 = blockIdx.y * 16;
    float* st = a.state + ((long long)h * DN + 16 * wave + 4 * g) * a.dv + c0 + m;
    deltax4_t S;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = a.pos0 > 0 ? st[(long long)r * a.dv] : 0.0f;
    // every wave requests the same number of pieces at addresses that only advance from chunk to chunk; a wave that has no use for them asks for one line
    struct Tile { deltap_t x[NS][3]; } tile[2];              // waves 0, 1: U' of the two token halves, 2, 3: W Q
    struct Rest { deltap_t ud[3], x[3]; float wc; } rest[2]; // x: V' of waves 0 and 1 (four floats), the outputs' product of waves 2 and 3
    const deltap_t* tp = (wave < 2 ? A.ut : A.qw) + ((long long)h * 2 + (wave & 1)) * NS * 192 + (wave < 4 ? lane : 0);
    const deltap_t* up = A.udt + ((long long)h * NW + wave) * 192 + lane;
    const deltap_t* xp = wave < 2 ? reinterpret_cast<const deltap_t*>(A.vt + ((long long)h * a.dv + c0 + m) * C + 16 * wave + 4 * g) : A.pm + ((long long)h * 2 + (wave & 1)) * 192 + (wave < 4 ? lane : 0);
    const long long xstep = (long long)a.H * (wave < 2 ? a.dv * C / 4 : 2 * 192);
    const int t1 = wave < 4 ? 64 : 0, x1 = wave == 2 || wave == 3 ? 64 : 0;
    auto request_tile = [&](Tile& o, int n) {
        const deltap_t* at = tp + (long long)n * a.H * 2 * NS * 192;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int i = 0; i < 3; ++i) o.x[s][i] = at[(3 * s + i) * t1];
    };
    auto request_rest = [&](Rest& o, int n) {
        const deltap_t *ud = up + (long long)n * a.H * NW * 192, *x = xp + n * xstep;
#pragma unroll
        for (int i = 0; i < 3; ++i) { o.ud[i] = ud[64 * i]; o.x[i] = x[x1 * i]; }
        o.wc = A.wc[(long long)n * a.H + h];
    };
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };   // (requests to memory stay under way)
    auto leave = [&](deltap_t (&to)[64], int half, uint32_t w0, uint32_t w1) { reinterpret_cast<uint2*>(&to[lane])[half] = uint2{w0, w1}; };
    const deltax4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    deltax4_t o;
    auto chunk = [&](Tile& t, Rest& cur, int ahead) {
        const DeltaPieces sp = delta_split(S);
#pragma unroll
        for (int i = 0; i < 3; ++i) leave(sb[i][wave / 2], wave & 1, sp.w[i][0], sp.w[i][1]);
        meet();
        deltax4_t sum = zero;
        if (wave < 4) {                                       // (uniform over the wave)
            deltax4_t small[2] = {zero, zero};
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const deltap_t y[3] = {sb[0][s][lane], sb[1][s][lane], sb[2][s][lane]};
                delta_mul(sum, small[s & 1], t.x[s], y);
            }
            sum += small[0] + small[1];
            if (wave < 2) {
                const DeltaPieces dp = delta_split(__builtin_bit_cast(deltax4_t, cur.x[0]) - sum);
#pragma unroll
                for (int i = 0; i < 3; ++i) leave(db[i], wave, dp.w[i][0], dp.w[i][1]);
            }
        }
        request_tile(t, ahead);
        meet();
        deltap_t d[3] = {db[0][lane], db[1][lane], db[2][lane]};
        deltax4_t small = zero;
        S *= cur.wc;
        delta_mul(S, small, cur.ud, d);
        S += small;
        if (wave == 2 || wave == 3) {
            // a token's output takes the d of the tokens before it only: zeros above the diagonal do not stop an infinity or a NaN, so such a d is taken out of
            // the product and every output from its token on is a NaN
            int bad = C;
#pragma unroll
            for (int j = 7; j >= 0; --j) {
                const uint32_t half = j & 1 ? 0xFFFF0000u : 0xFFFFu;
                if ((d[0][j / 2] & half & 0x7F807F80u) == (half & 0x7F807F80u)) { bad = delta_place(g, j); d[0][j / 2] &= ~half; }
            }
            if (__ballot(bad < C)) {
                bad = min(bad, __shfl_xor(bad, 16, 64));
                bad = min(bad, __shfl_xor(bad, 32, 64));
            }
            small = zero;
            delta_mul(sum, small, cur.x, d);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = 16 * (wave - 2) + 4 * g + r >= bad ? NAN : sum[r] + small[r];
        }
        request_rest(cur, ahead);
    };
    // a chunk's outputs are stored at the next one's start: the wait for its operands also waits for the stores before them, which are then long gone
    auto store = [&](int n) {
        if (wave != 2 && wave != 3) return;
        float* p = a.out + (long long)n * C * a.ldo + (long long)h * a.dv + c0 + m;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (wave - 2) + 4 * g + r;
            if (n * C + row < a.T) p[(long long)row * a.ldo] = o[r];
        }
    };
    const int last = A.chunks - 1;
#pragma unroll
    for (int u = 0; u < 2; ++u) { request_tile(tile[u], min(u, last)); request_rest(rest[u], min(u, last)); }
    for (int n = 0; n <= last; n += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (n + u > last) break;
            if (n + u) store(n + u - 1);
            chunk(tile[u], rest[u], min(n + u + 2, last));
        }
    }
    store(A.chunks - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) st[(long long)r * a.dv] = S[r];
}

// The chunks take portions whose rows can be read four floats at a time (150 tokens of the heads above: 33 us against 100); everything else walks token by token.
// From a chunk and a half on: the two launches take 17 - 25 us however short the portion is (us, walk / chunks: 32 tokens of 16 heads of 128 x 128 20.1 / 21.9, 33: 21.6 / 23.9, 48:
// 26.3 / 24.1, 64: 32.9 / 24.5; 64 x 128 15.3 / 17.7, 48: 19.7 / 19.0), from two on with wider values, whose substitution goes more than one round (256: 48 tokens 24.8 / 29.6, 64: 30.8 / 30.1).
inline bool delta_chunked(const RecArgs& a) {
    return a.az && a.head_gates && a.write_gated && a.unit_k && !a.conv_w && a.T >= (a.dv > 128 ? 2 * kDeltaChunk : kDeltaChunk * 3 / 2) && (a.dn == 64 || a.dn == 128) && a.dv % 16 == 0 && a.ldq % 4 == 0 && a.ldk % 4 == 0 &&
           !(((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.packed) & 15) && a.H <= 65535;
}

template <int DN>
static int launch_delta_chunks(const RecArgs& a, hipStream_t s) {
    DeltaArgs A{a, (a.T + kDeltaChunk - 1) / kDeltaChunk};
    const size_t blocks = (size_t)A.chunks * a.H;
    A.vt = a.packed;
    A.ut = reinterpret_cast<deltap_t*>(A.vt + blocks * kDeltaChunk * a.dv);
    A.qw = A.ut + blocks * (DN / 16) * 192;
    A.udt = A.qw + blocks * (DN / 16) * 192;
    A.pm = A.udt + blocks * (DN / 16) * 192;
    A.wc = reinterpret_cast<float*>(A.pm + blocks * 2 * 192);
    hipLaunchKernelGGL(delta_chunk_solve_kernel<DN>, dim3(A.chunks, a.H), dim3(256), 0, s, A);
    const int st = last_launch_status();
    if (st != NTK_OK) return st;
    hipLaunchKernelGGL(delta_chunk_walk_kernel<DN>, dim3(a.H, a.dv / 16), dim3(4 * DN), 0, s, A);
    return last_launch_status();
}

}  // namespace ntk
