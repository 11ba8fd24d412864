// moe_route.hip.h -- a token's router scores and choice by one workgroup: a launch of its own (moe.hip), or beside the attention of decoded tokens (latent_attention.hip).
#pragma once
#include "common.hip.h"
#include "../../include/ntk_layers.h"

namespace ntk {

constexpr int kMaxExperts = 256;

struct RouteForm { int score, groups, keep, group_top, renorm; float scale; const float* correction; const float* add_y; int ld_add; const float* add_w; float add_eps;
    const float* src; int ldsrc; const float* norm_w; float norm_eps, norm_offset;     // (norm_w: the token's row is the RMS norm of a row of src, formed in the launch and left in h; NULL: h holds it)
};

// the largest of a wave's 4 x 64 values (lane l holds entries l, l + 64, l + 128, l + 192); equal values: the lower index
__device__ __forceinline__ void wave_argmax4(const float (&v)[4], int lane, float& bv, int& bi) {
    bv = wave_max(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    bi = 0;
#pragma unroll
    for (int c = 3; c >= 0; --c) {                            // (the lowest index is the first lane of the first quarter that holds the value)
        const unsigned long long m = __ballot(v[c] == bv);
        if (m) bi = 64 * c + __ffsll((unsigned long long)m) - 1;
    }
}

// scores and the picks by one wave: lane l holds experts l, l + 64, l + 128, l + 192; z [E] in LDS
__device__ __forceinline__ void pick_experts(float* z, int lane, long long t, int E, int top, const RouteForm& f, int* ids, float* wts) {
    float v[4];
    float den = 1.0f;
    if (f.score == 0) {
        float m = -INFINITY;
#pragma unroll
        for (int c = 0; c < 4; ++c) { v[c] = lane + 64 * c < E ? z[lane + 64 * c] : -INFINITY; m = fmaxf(m, v[c]); }
        m = wave_max(m);
        den = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) { v[c] = lane + 64 * c < E ? expf(v[c] - m) : -INFINITY; den += fmaxf(v[c], 0.0f); }
        den = wave_sum(den);
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = lane + 64 * c < E ? 1.0f / (1.0f + expf(-z[lane + 64 * c])) : -INFINITY;
    }
    if (f.correction) {     // (uniform) what is chosen by is no longer what is weighted with: the scores stay in LDS, v becomes the choice scores
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (lane + 64 * c < E) { const float s = v[c] / den; z[lane + 64 * c] = s; v[c] = s + f.correction[lane + 64 * c]; }
        __builtin_amdgcn_wave_barrier();
    }
    __shared__ int pick_id[kMaxExperts];
    __shared__ float pick_sc[kMaxExperts];
    if (f.groups > 1) {
        // group scores: lane l owns groups l, l + 64, ...: the sum of the group's `group_top` largest scores
        __shared__ float sc[kMaxExperts];
        __shared__ unsigned char open_group[kMaxExperts];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (lane + 64 * c < E) sc[lane + 64 * c] = v[c];
        __builtin_amdgcn_wave_barrier();
        const int per = E / f.groups;
        float gs[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int g = lane + 64 * c;
            gs[c] = -INFINITY;
            if (g < f.groups) {
                float sum = 0.0f;
                const int nt = min(f.group_top, per);
                float last = INFINITY;
                int last_e = -1;
                for (int k = 0; k < nt; ++k) {                // the largest behind the one before it (equal values: by index)
                    float best = -INFINITY;
                    int bi = -1;
                    for (int e = g * per; e < (g + 1) * per; ++e)
                        if ((sc[e] < last || (sc[e] == last && e > last_e)) && sc[e] > best) { best = sc[e]; bi = e; }
                    last = best;
                    last_e = bi;
                    sum += best;
                }
                gs[c] = sum;
            }
            if (g < kMaxExperts) open_group[g] = 0;
        }
        __builtin_amdgcn_wave_barrier();
        for (int k = 0; k < f.keep; ++k) {                    // (taken ones are marked -inf)
            float bv;
            int bi;
            wave_argmax4(gs, lane, bv, bi);
            if (lane == 0) open_group[bi] = 1;
            if ((bi & 63) == lane) gs[bi >> 6] = -INFINITY;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (lane + 64 * c < E && !open_group[(lane + 64 * c) / per]) v[c] = -INFINITY;
    }
    float chosen = 0.0f;
    for (int s = 0; s < top; ++s) {
        float bv;
        int bi;
        wave_argmax4(v, lane, bv, bi);
        const float sc1 = f.correction ? z[bi] : bv / den;
        chosen += sc1;
        if (lane == 0) { pick_id[s] = bi; pick_sc[s] = sc1; }
        if ((bi & 63) == lane) v[bi >> 6] = -INFINITY;
    }
    const float mul = (f.renorm ? 1.0f / (chosen + 1e-20f) : 1.0f) * f.scale;
    for (int s = lane; s < top; s += 64) { ids[t * top + s] = pick_id[s]; wts[t * top + s] = pick_sc[s] * mul; }   // (same wave wrote them: in order)
}

struct RouteJob { int* ids; float* wts; float* sgate; float* h; int ldh; const float* wr; const float* wsg; int n, E, top; RouteForm f; };
// checks what ntk_moe_norm_route checks; NTK_OK: *job is complete
int norm_route_job(const ntk_norm_route* d, RouteJob* job);

// One token: the WAVES waves share the experts (wave w: experts w, w + WAVES, ...), EA rows of the router at a time and four requests of each before any is used, the first of them under the row's norm (EA > 1); the first wave then does the
// softmax and the `top` picks over the scores in LDS.  xs [n]: the token's row in LDS, on 16 bytes.  Latency bounds it: the row, its norm, the router's rows, the picks, one after the other.
// EA > 1 costs registers: for a few tokens, not for the many of a prompt, whose workgroups are to share a CU.
template <int WAVES, int EA>
__device__ __forceinline__ void route_token(const RouteJob& j, long long t, float* xs) {
    constexpr int THREADS = 64 * WAVES;
    __shared__ float z[kMaxExperts];
    __shared__ float red[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = j.n, E = j.E;
    const RouteForm& f = j.f;
    float* x = j.h + t * j.ldh;
    const bool vec = (n % 4 == 0) && !((uintptr_t)j.wr & 15) && !(j.wsg && ((uintptr_t)j.wsg & 15));
    const int rows = E + (j.wsg ? 1 : 0);
    auto row = [&](int e) { return e < E ? j.wr + (long long)e * n : j.wsg; };
    constexpr int KA = 4;
    float4 a[EA][KA];
    auto request = [&](int e0, int k0) {                     // (rows and columns past the end: zeros)
#pragma unroll
        for (int i = 0; i < EA; ++i) {
            const int e = e0 + i * WAVES;
            const float* w = row(min(e, rows - 1));
#pragma unroll
            for (int u = 0; u < KA; ++u) a[i][u] = k0 + 256 * u < n && e < rows ? *reinterpret_cast<const float4*>(w + k0 + 256 * u) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    if (EA > 1 && vec) request(wave, lane * 4);              // (under the row's way here and its norm)
    if (f.norm_w) {    // (uniform).  us, one token of 2048 among 32 experts: 6.4 the norm in a launch of its own and 7.5 the choice, 9.1 so (weights requested ahead of the row: 10.9)
        const float* y = f.src + t * f.ldsrc;
        float ss = 0.0f;
        constexpr int NA = EA > 1 ? 4 : 1;                   // weights of the norm that are requested with the row
        float nw[NA];
        if (EA > 1)
#pragma unroll
            for (int u = 0; u < NA; ++u) nw[u] = (int)threadIdx.x + THREADS * u < n ? f.norm_w[threadIdx.x + THREADS * u] : 0.0f;
        for (int k = threadIdx.x; k < n; k += THREADS) { const float v = y[k]; xs[k] = v; ss = fmaf(v, v, ss); }
        const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + f.norm_eps);
        if (EA > 1)
#pragma unroll
            for (int u = 0; u < NA; ++u) {
                const int k = threadIdx.x + THREADS * u;
                if (k >= n) break;
                const float v = xs[k] * inv * (f.norm_offset + nw[u]);
                xs[k] = v;
                x[k] = v;
            }
        for (int k = threadIdx.x + (EA > 1 ? NA * THREADS : 0); k < n; k += THREADS) {
            const float v = xs[k] * inv * (f.norm_offset + f.norm_w[k]);
            xs[k] = v;
            x[k] = v;
        }
    } else if (f.add_y) {     // (uniform) what the row is still owed joins it: y / rms(y) * w; a thread re-reads its own entries
        const float* y = f.add_y + t * f.ld_add;
        float ss = 0.0f;
        for (int k = threadIdx.x; k < n; k += THREADS) { xs[k] = x[k]; ss = fmaf(y[k], y[k], ss); }
        const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)n + f.add_eps);
        for (int k = threadIdx.x; k < n; k += THREADS) {
            const float v = fmaf(y[k] * inv, f.add_w[k], xs[k]);
            xs[k] = v;
            x[k] = v;
        }
    } else {
        for (int k = threadIdx.x; k < n; k += THREADS) xs[k] = x[k];
    }
    __syncthreads();
    auto leave = [&](int e, float s) {
        s = wave_sum(s);
        if (lane != 0) return;
        if (e < E) z[e] = s;
        else if (j.sgate) j.sgate[t] = 1.0f / (1.0f + expf(-s));
    };
    if (vec && EA == 1) {
        for (int e = wave; e < rows; e += WAVES) {
            const float* w = row(e);
            float s = 0.0f;
#pragma unroll 4
            for (int k = lane * 4; k < n; k += 256) {
                const float4 a4 = *reinterpret_cast<const float4*>(w + k), x4 = *reinterpret_cast<const float4*>(xs + k);
                s = fmaf(a4.x, x4.x, s); s = fmaf(a4.y, x4.y, s); s = fmaf(a4.z, x4.z, s); s = fmaf(a4.w, x4.w, s);
            }
            leave(e, s);
        }
    } else if (vec) {
        for (int e0 = wave; e0 < rows; e0 += EA * WAVES) {       // (uniform over the wave)
            float s[EA];
#pragma unroll
            for (int i = 0; i < EA; ++i) s[i] = 0.0f;
            for (int k0 = lane * 4; k0 < n; k0 += 256 * KA) {
                if (e0 > wave || k0 > lane * 4) request(e0, k0);
#pragma unroll
                for (int u = 0; u < KA; ++u) {
                    if (k0 + 256 * u >= n) break;
                    const float4 x4 = *reinterpret_cast<const float4*>(xs + k0 + 256 * u);
#pragma unroll
                    for (int i = 0; i < EA; ++i) {
                        s[i] = fmaf(a[i][u].x, x4.x, s[i]); s[i] = fmaf(a[i][u].y, x4.y, s[i]); s[i] = fmaf(a[i][u].z, x4.z, s[i]); s[i] = fmaf(a[i][u].w, x4.w, s[i]);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < EA; ++i)
                if (e0 + i * WAVES < rows) leave(e0 + i * WAVES, s[i]);
        }
    } else {
        for (int e = wave; e < rows; e += WAVES) {
            const float* w = row(e);
            float s = 0.0f;
            for (int k = lane; k < n; k += 64) s = fmaf(w[k], xs[k], s);
            leave(e, s);
        }
    }
    __syncthreads();
    if (wave != 0) return;
    pick_experts(z, lane, t, E, j.top, f, j.ids, j.wts);
}

}  // namespace ntk
