// delta_chunk.hip.h -- the delta rule with one gate per head, 32 tokens at a time on the F32 matrix instructions.  Included by gated_recurrence.hip.
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
// and 16 value columns (delta_chunk_walk_kernel), the state in the accumulators of its waves all the way.  1024 tokens of 16 heads of 128 x 128: 93 us, where the walk
// token by token, its pre-pass and the settling of its segments took 277.
#pragma once

namespace ntk {

constexpr int kDeltaChunk = 32;
typedef float deltax4_t __attribute__((ext_vector_type(4)));

struct DeltaArgs {
    RecArgs r;
    int chunks;
    float *vt, *ut, *qw, *udt, *pm, *wc;   // per (chunk, head): [dv][32], [32][dn], [32][dn], [dn][32], [32][32], one number
};

// floats of DeltaArgs' buffers
inline size_t delta_chunk_floats(int T, int H, int dn, int dv) {
    const size_t blocks = (size_t)((T + kDeltaChunk - 1) / kDeltaChunk) * H;
    return blocks * ((size_t)kDeltaChunk * (dv + 3 * dn + kDeltaChunk) + 4);
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
    float* pm = A.pm + blk * C * C;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tile = wave + 4 * u, ti = tile % 3 > 0, tj = tile % 3 == 2, s = 16 * tj + m;
        if (tile >= 6) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * ti + 4 * g + r;
            if (tile < 3) am[t * LA + s] = s < t ? av[t] * rm[t][s] * acc[u][r] : 0.0f;
            else pm[t * C + s] = s <= t ? rm[t][s] * acc[u][r] : 0.0f;
        }
    }
    pm[(tid / 16) * C + 16 + tid % 16] = 0.0f;                // the tile above the diagonal (256 threads: 16 x 16)
    __syncthreads();
    // W q, and the keys with what decays behind them, a channel's 32 tokens in a row
#pragma unroll 2
    for (int e = tid; e < C * DN / 4; e += 256) {
        const int t = e / (DN / 4), d = e % (DN / 4) * 4;
        const float4 q4 = *reinterpret_cast<const float4*>(qs + t * LD + d);
        *reinterpret_cast<float4*>(A.qw + blk * C * DN + 4 * e) = float4{cw[t] * q4.x, cw[t] * q4.y, cw[t] * q4.z, cw[t] * q4.w};
    }
#pragma unroll 2
    for (int e = tid; e < C * DN / 4; e += 256) {
        const int t = e % (C / 4) * 4, d = e / (C / 4);
        const float* u = us + t * LD + d;
        const float* w = rm[C - 1] + t;
        *reinterpret_cast<float4*>(A.udt + blk * C * DN + 4 * e) = float4{w[0] * u[0], w[1] * u[LD], w[2] * u[2 * LD], w[3] * u[3 * LD]};
    }
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
                for (int i = 0; i < 4; ++i) A.ut[(blk * C + t + i) * DN + c - a.dv] = x[i];
        }
    }
}

// grid (H, dv / 16) -- the column blocks of a head, which read the same operands, fall on the same L2 where H is a multiple of the eight --, a wave per 16 key channels.  Wave w's accumulators are rows 16 w ... of the 16 columns of the state; a matrix instruction's four k entries may be
// any four as long as both operands agree, so register r of the accumulators (rows 16 w + 4 g + r of lane group g) is the state's operand as it stands.  Per chunk:
// every wave's share of U' S_0 and W Q S_0 meets in LDS, one wave per 16 x 16 tile of the two sums it, D = V' - U' S_0 goes to all, then the state's update everywhere
// and the outputs' product with D in two waves.  Bound by this chain (two barriers a chunk, 1600 of 5200 cycles in matrix instructions); operands are requested two
// chunks ahead (one: 76 us instead of 72 for 1024 tokens of 16 heads of 128 x 128).
template <int DN>
__global__ __launch_bounds__(4 * DN, DN / 64) void delta_chunk_walk_kernel(const DeltaArgs A) {
    constexpr int C = kDeltaChunk, NW = DN / 16, LD = 18;     // (18: the four lane groups' rows of D fall into different banks)
    static_assert(NW >= 4, "a wave per summed tile");
    __shared__ __attribute__((aligned(16))) deltax4_t part[NW][4][64];
    __shared__ float dl[C * LD];
    const RecArgs& a = A.r;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const int h = blockIdx.x, c0 = blockIdx.y * 16;
    float* st = a.state + ((long long)h * DN + 16 * wave + 4 * g) * a.dv + c0 + m;
    deltax4_t S;
#pragma unroll
    for (int r = 0; r < 4; ++r) S[r] = a.pos0 > 0 ? st[(long long)r * a.dv] : 0.0f;
    // x: V' of waves 0 and 1, the outputs' product of waves 2 and 3; every wave requests the same number of pieces at addresses that only advance from chunk to chunk
    struct Operands { deltax4_t ut[2], qw[2], ud[2], x[2]; float wc; } op[3];
    const long long b0 = h, xstep = (long long)a.H * C * (wave < 2 ? a.dv : C);
    const float* utp = A.ut + (b0 * C + m) * DN + 16 * wave + 4 * g;
    const float* qwp = A.qw + (b0 * C + m) * DN + 16 * wave + 4 * g;
    const float* udp = A.udt + (b0 * DN + 16 * wave + m) * C + 8 * g;
    const float* xp = wave < 2 ? A.vt + (b0 * a.dv + c0 + m) * C + 16 * wave + 4 * g : A.pm + (b0 * C + 16 * (wave & 1) + m) * C + 8 * g;
    const int x1 = wave < 2 ? 0 : 4;
    auto request = [&](Operands& o, int n) {
        const long long at = (long long)n * a.H * C * DN;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            o.ut[i] = *reinterpret_cast<const deltax4_t*>(utp + at + 16 * i * DN);
            o.qw[i] = *reinterpret_cast<const deltax4_t*>(qwp + at + 16 * i * DN);
            o.ud[i] = *reinterpret_cast<const deltax4_t*>(udp + at + 4 * i);
            o.x[i] = *reinterpret_cast<const deltax4_t*>(xp + n * xstep + i * x1);
        }
        o.wc = A.wc[(long long)n * a.H + h];
    };
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };   // (requests to memory stay under way)
    deltax4_t o;
    auto chunk = [&](const Operands& cur) {
        deltax4_t p[4] = {};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                p[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.ut[i][r], S[r], p[i], 0, 0, 0);
                p[2 + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.qw[i][r], S[r], p[2 + i], 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][i][lane] = p[i];
        meet();
        deltax4_t sum = {};
        if (wave < 4) {                                       // (uniform over the wave)
            deltax4_t q[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) q[w] = part[w][wave][lane];
#pragma unroll
            for (int w = 0; w < NW; ++w) sum += q[w];
            if (wave < 2)
#pragma unroll
                for (int r = 0; r < 4; ++r) dl[(16 * wave + 4 * g + r) * LD + m] = cur.x[0][r] - sum[r];
        }
        meet();
        float d[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) d[j] = dl[(8 * g + j) * LD + m];
        S *= cur.wc;
#pragma unroll
        for (int j = 0; j < 8; ++j) S = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.ud[j / 4][j % 4], d[j], S, 0, 0, 0);
        if (wave == 2 || wave == 3) {
            // a token's output takes the d of the tokens before it only: zeros above the diagonal do not stop an infinity or a NaN, so such a d is taken out of
            // the product and every output from its token on is a NaN
            int bad = C;
#pragma unroll
            for (int j = 7; j >= 0; --j)
                if (!(fabsf(d[j]) < INFINITY)) { bad = 8 * g + j; d[j] = 0.0f; }
            if (__ballot(bad < C)) {
                bad = min(bad, __shfl_xor(bad, 16, 64));
                bad = min(bad, __shfl_xor(bad, 32, 64));
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.x[j / 4][j % 4], d[j], sum, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = 16 * (wave - 2) + 4 * g + r >= bad ? NAN : sum[r];
        }
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
    request(op[0], 0);
    request(op[1], min(1, last));
    for (int n = 0; n <= last; n += 3) {
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            if (n + u > last) break;
            if (n + u) store(n + u - 1);
            request(op[(u + 2) % 3], min(n + u + 2, last));
            chunk(op[u]);
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
    A.ut = A.vt + blocks * kDeltaChunk * a.dv;
    A.qw = A.ut + blocks * kDeltaChunk * DN;
    A.udt = A.qw + blocks * kDeltaChunk * DN;
    A.pm = A.udt + blocks * kDeltaChunk * DN;
    A.wc = A.pm + blocks * kDeltaChunk * kDeltaChunk;
    hipLaunchKernelGGL(delta_chunk_solve_kernel<DN>, dim3(A.chunks, a.H), dim3(256), 0, s, A);
    const int st = last_launch_status();
    if (st != NTK_OK) return st;
    hipLaunchKernelGGL(delta_chunk_walk_kernel<DN>, dim3(a.H, a.dv / 16), dim3(4 * DN), 0, s, A);
    return last_launch_status();
}

}  // namespace ntk
