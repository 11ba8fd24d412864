// moe.hip -- the routing side of a mixture of experts: router scores and the choice (F32; optionally by score plus a learned correction, optionally among the best groups
// only; in one launch, or the choice alone behind a product), the stable grouping of (token, slot) pairs by expert that
// the grouped product (dense.hip) consumes, the clipped gated activation between an expert's two products, and the weighted sum (identity experts: of the input itself) back into the
// residual stream.  The experts' products themselves are ntk_dense calls over the stacked expert matrices.
//
// A token's result never depends on the other tokens of the launch: the grouping only decides WHERE a pair's row sits, each row is computed on its
// own, and the sum over a token's slots runs in slot order.
#include "moe_route.hip.h"

namespace ntk {

// one workgroup per token
constexpr int kRouteWaves = 16;
__global__ __launch_bounds__(64 * kRouteWaves) void moe_route_kernel(const RouteJob j) {
    extern __shared__ __attribute__((aligned(16))) float xs[];   // the token's row
    route_token<kRouteWaves, 1>(j, blockIdx.x, xs);
}

// the same picks from logits that a product left: z [T][ldz] = [E router outputs | the shared unit's gate (if sgate)], one wave per token
__global__ __launch_bounds__(64) void moe_pick_kernel(int* ids, float* wts, float* sgate, const float* zg, int ldz, int E, int top, const RouteForm f) {
    __shared__ float z[kMaxExperts];
    const int lane = threadIdx.x;
    const long long t = blockIdx.x;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (lane + 64 * c < E) z[lane + 64 * c] = zg[t * ldz + lane + 64 * c];
    if (sgate && lane == 0) sgate[t] = 1.0f / (1.0f + expf(-zg[t * ldz + E]));
    __syncthreads();
    pick_experts(z, lane, t, E, top, f, ids, wts);
}

// Stable counting sort of the pairs by expert, one workgroup: each of its 16 waves takes a contiguous run of pairs, 64 at a time, one a lane.  The lanes that hold
// the same expert find each other by one ballot per bit of the index, so a lane's rank among them is a bit count and one lane of each expert keeps the wave's count;
// a scan in (expert, wave) order gives every wave its first row of each expert, and it goes through its run once more to place the pairs.  A chain of latencies
// whatever the form: a thread per (expert, segment) that looked at its segment pair by pair issued a store per pair and expert, 42 us at 6144 pairs of 32
// experts (27 with the ids read four at a time), 9 so.
constexpr int kGroupThreads = 1024, kGroupWaves = kGroupThreads / 64, kGroupAhead = 8;
__global__ __launch_bounds__(kGroupThreads) void moe_group_kernel(int* offsets, int* order, int* where, const int* __restrict__ ids, int n_pairs, int E, int bits) {
    __shared__ int cnt[kMaxExperts * kGroupWaves];                // [expert][wave]; E < 256
    __shared__ int wave_total[kGroupWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < kMaxExperts * kGroupWaves; i += kGroupThreads) cnt[i] = 0;
    __syncthreads();
    const int per = ((n_pairs + kGroupWaves - 1) / kGroupWaves + 63) & ~63;
    const int i0 = min(wave * per, n_pairs), i1 = min(i0 + per, n_pairs);
    // visit(pair, expert, rank among the chunk's pairs of this expert, how many they are)
    auto walk = [&](auto&& visit) {
        for (int g = i0; g < i1; g += 64 * kGroupAhead) {         // (uniform over the wave)
            int id[kGroupAhead];
#pragma unroll
            for (int c = 0; c < kGroupAhead; ++c) { const int i = g + 64 * c + lane; id[c] = i < i1 ? ids[i] : -1; }
#pragma unroll
            for (int c = 0; c < kGroupAhead; ++c) {
                if (g + 64 * c >= i1) break;
                const bool valid = (unsigned)id[c] < (unsigned)E;
                unsigned long long same = __ballot(valid);
                for (int b = 0; b < bits; ++b) {
                    const bool one = (id[c] >> b) & 1;
                    const unsigned long long m = __ballot(one);
                    same &= one ? m : ~m;
                }
                if (valid) visit(g + 64 * c + lane, id[c], __popcll(same & ((1ull << lane) - 1)), __popcll(same));
                __builtin_amdgcn_wave_barrier();
            }
        }
    };
    walk([&](int, int e, int rank, int n) { if (rank == 0) cnt[e * kGroupWaves + wave] += n; });
    __syncthreads();
    {   // exclusive scan of the E * 16 counts, four in a row to a thread
        int c[4], mine = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) { c[k] = cnt[4 * tid + k]; mine += c[k]; }
        int inc = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(inc, o, 64);
            if (lane >= o) inc += up;
        }
        if (lane == 63) wave_total[wave] = inc;
        __syncthreads();
        int at = inc - mine;
        for (int k = 0; k < wave; ++k) at += wave_total[k];
        if (tid % (kGroupWaves / 4) == 0 && tid / (kGroupWaves / 4) <= E) offsets[tid / (kGroupWaves / 4)] = at;     // (an expert's first wave; E itself: the sum of all)
#pragma unroll
        for (int k = 0; k < 4; ++k) { cnt[4 * tid + k] = at; at += c[k]; }
    }
    __syncthreads();
    walk([&](int i, int e, int rank, int n) {
        int* at = cnt + e * kGroupWaves + wave;
        const int to = *at + rank;
        order[to] = i;
        where[i] = to;
        __builtin_amdgcn_wave_barrier();
        if (rank == 0) *at += n;                                  // (the wave's lanes have read it: in order)
    });
}

// V outputs a thread; bound by the rows it reads and writes.  6144 rows of 1408: 30 us with one output a thread, 19 with four.
template <int V>
__global__ void clipped_glu_kernel(float* a, int lda, const float* gu, int ldgu, int ff, float limit, float alpha, float cubic, float up_offset) {
    struct __attribute__((aligned(4 * V))) Vec { float v[V]; };
    const long long r = blockIdx.y;
    const int f = (blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (f >= ff) return;
    const Vec gate = *reinterpret_cast<const Vec*>(gu + r * ldgu + f), up = *reinterpret_cast<const Vec*>(gu + r * ldgu + ff + f);
    Vec o;
#pragma unroll
    for (int c = 0; c < V; ++c) {
        const float g = fminf(gate.v[c], limit);
        const float u = fminf(fmaxf(up.v[c], -limit), limit);
        const float z = cubic != 0.0f ? fmaf(cubic * g * g, g, g) : g;
        o.v[c] = g * (1.0f / (1.0f + expf(-alpha * z))) * (u + up_offset);
    }
    *reinterpret_cast<Vec*>(a + r * lda + f) = o;
}

// out[t] = the chosen rows times their weights, in slot order, + the shared unit's times its gate (+ mix, + what is there); V columns a thread.  Bound by the rows
// it reads; the requests of kCombineSlots slots are under way together, and four columns a thread where the rows allow it: 26 us -> 14.5 at 1024 tokens of six
// choices of 2048 (one column a thread, slot by slot).
constexpr int kCombineSlots = 4;
template <bool ADD, int V>
__global__ void moe_combine_kernel(float* x, const float* mix, const float* d, const int* where, const float* wts, const float* shared, const float* sgate,
                                   int top, int n, const int* ids, int n_experts, const float* h, int ldh) {
    struct __attribute__((aligned(4 * V))) Vec { float v[V]; };
    const long long t = blockIdx.y;
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (i >= n) return;
    auto at = [&](const float* p) { return *reinterpret_cast<const Vec*>(p + i); };
    Vec sh{}, mx{}, s{}, row[kCombineSlots];
    if (shared) sh = at(shared + t * n);
    if (mix) mx = at(mix + t * n);
    if constexpr (ADD) row[0] = at(x + t * n);
    const Vec was = row[0];
    for (int k0 = 0; k0 < top; k0 += kCombineSlots) {
#pragma unroll
        for (int j = 0; j < kCombineSlots; ++j) {
            const long long p = t * top + min(k0 + j, top - 1);
            row[j] = at(ids && ids[p] >= n_experts ? h + t * ldh : d + (long long)(where ? where[p] : p) * n);   // an identity expert gives the input back
        }
#pragma unroll
        for (int j = 0; j < kCombineSlots; ++j) {
            if (k0 + j >= top) break;
            const float w = wts[t * top + k0 + j];
#pragma unroll
            for (int c = 0; c < V; ++c) s.v[c] = fmaf(w, row[j].v[c], s.v[c]);
        }
    }
    const float g = shared && sgate ? sgate[t] : 1.0f;
#pragma unroll
    for (int c = 0; c < V; ++c) {
        if (shared) s.v[c] = fmaf(g, sh.v[c], s.v[c]);
        if (mix) s.v[c] += mx.v[c];
        if constexpr (ADD) s.v[c] = was.v[c] + s.v[c];
    }
    *reinterpret_cast<Vec*>(x + t * n + i) = s;
}

template <bool ADD>
static int launch_combine(float* x, const float* mix, const float* d, const int* where, const float* wts, const float* shared, const float* sgate, int T, int top, int n,
                          const int* ids, int n_experts, const float* h, int ldh, hipStream_t s) {
    const bool vec = n % 4 == 0 && !(((uintptr_t)x | (uintptr_t)mix | (uintptr_t)d | (uintptr_t)shared) & 15) && !(ids && (((uintptr_t)h & 15) || ldh % 4));
    if (vec) hipLaunchKernelGGL((moe_combine_kernel<ADD, 4>), dim3((n / 4 + 255) / 256, T), dim3(256), 0, s, x, mix, d, where, wts, shared, sgate, top, n, ids, n_experts, h, ldh);
    else hipLaunchKernelGGL((moe_combine_kernel<ADD, 1>), dim3((n + 255) / 256, T), dim3(256), 0, s, x, mix, d, where, wts, shared, sgate, top, n, ids, n_experts, h, ldh);
    return last_launch_status();
}

}  // namespace ntk

using namespace ntk;

int ntk_moe_route(int* ids, float* wts, float* sgate, const float* h, int ldh, const float* w_router, const float* shared_gate_w, int T, int n, int E, int top,
                  void* stream) {
    ntk_route_desc r{};
    r.groups = r.keep = r.group_top = r.renorm = 1;
    r.scale = 1.0f;   // softmax scores, no groups, weights renormalised over the chosen
    return ntk_moe_route_ex(ids, wts, sgate, h, ldh, w_router, shared_gate_w, T, n, E, top, &r, stream);
}

static int route_form(const ntk_route_desc* r, int E, int top, RouteForm* f) {
    if (r->score != 0 && r->score != 1) return NTK_E_SHAPE;
    const int groups = r->groups > 1 ? r->groups : 1;
    if (groups > 1 && (E % groups || r->keep < 1 || r->keep > groups || r->group_top < 1 || r->group_top > 8 || (long long)r->keep * (E / groups) < top)) return NTK_E_SHAPE;
    *f = RouteForm{r->score, groups, r->keep, r->group_top, r->renorm, r->scale, r->correction, r->add_y, r->ld_add, r->add_w, r->add_eps, nullptr, 0, nullptr, 0.0f, 0.0f};
    return NTK_OK;
}

int ntk_moe_route_ex(int* ids, float* wts, float* sgate, const float* h, int ldh, const float* w_router, const float* shared_gate_w, int T, int n, int E, int top,
                     const ntk_route_desc* r, void* stream) {
    if (!ids || !wts || !h || !w_router || !r) return NTK_E_NULL;
    if (T < 0 || n <= 0 || E <= 0 || E > kMaxExperts || top <= 0 || top > E || ldh < n) return NTK_E_SHAPE;
    if (r->add_y && (!r->add_w || r->ld_add < n || r->add_y == h)) return NTK_E_SHAPE;
    if ((size_t)n * 4 > 128 * 1024) return NTK_E_SHAPE;
    RouteForm f;
    const int st = route_form(r, E, top, &f);
    if (st != NTK_OK || T == 0) return st;
    const RouteJob j{ids, wts, sgate, (float*)h, ldh, w_router, shared_gate_w, n, E, top, f};
    hipLaunchKernelGGL(moe_route_kernel, dim3(T), dim3(64 * kRouteWaves), (size_t)n * 4, resolve_stream(stream), j);
    return last_launch_status();
}

int ntk::norm_route_job(const ntk_norm_route* d, RouteJob* job) {
    if (!d || !d->ids || !d->wts || !d->h || !d->x || !d->norm_w || !d->w_router || !d->form) return NTK_E_NULL;
    if (d->T < 0 || d->n <= 0 || d->E <= 0 || d->E > kMaxExperts || d->top <= 0 || d->top > d->E || d->ldh < d->n || d->ldx < d->n || d->form->add_y || d->h == d->x) return NTK_E_SHAPE;
    if ((size_t)d->n * 4 > 128 * 1024) return NTK_E_SHAPE;
    RouteForm f;
    const int st = route_form(d->form, d->E, d->top, &f);
    if (st != NTK_OK) return st;
    f.src = d->x; f.ldsrc = d->ldx; f.norm_w = d->norm_w; f.norm_eps = d->norm_eps; f.norm_offset = d->norm_offset;
    *job = RouteJob{d->ids, d->wts, d->sgate, d->h, d->ldh, d->w_router, d->shared_gate_w, d->n, d->E, d->top, f};
    return NTK_OK;
}

int ntk_moe_norm_route(int* ids, float* wts, float* sgate, float* h, int ldh, const float* x, int ldx, const float* norm_w, float norm_eps, float norm_offset, const float* w_router,
                       const float* shared_gate_w, int T, int n, int E, int top, const ntk_route_desc* r, void* stream) {
    const ntk_norm_route d{ids, wts, sgate, h, ldh, x, ldx, norm_w, norm_eps, norm_offset, w_router, shared_gate_w, T, n, E, top, r};
    RouteJob j;
    const int st = norm_route_job(&d, &j);
    if (st != NTK_OK || T == 0) return st;
    hipLaunchKernelGGL(moe_route_kernel, dim3(T), dim3(64 * kRouteWaves), (size_t)n * 4, resolve_stream(stream), j);
    return last_launch_status();
}

int ntk_moe_pick(int* ids, float* wts, float* sgate, const float* z, int ldz, int T, int E, int top, const ntk_route_desc* r, void* stream) {
    if (!ids || !wts || !z || !r) return NTK_E_NULL;
    if (T < 0 || E <= 0 || E > kMaxExperts || top <= 0 || top > E || ldz < E + (sgate ? 1 : 0) || r->add_y) return NTK_E_SHAPE;
    RouteForm f;
    const int st = route_form(r, E, top, &f);
    if (st != NTK_OK || T == 0) return st;
    hipLaunchKernelGGL(moe_pick_kernel, dim3(T), dim3(64), 0, resolve_stream(stream), ids, wts, sgate, z, ldz, E, top, f);
    return last_launch_status();
}

int ntk_moe_group(int* offsets, int* order, int* where, const int* ids, int T, int top, int E, void* stream) {
    if (!offsets || !order || !where || !ids) return NTK_E_NULL;
    if (T < 0 || top <= 0 || E <= 0 || E >= 256) return NTK_E_SHAPE;
    int bits = 0;
    while ((1 << bits) < E) ++bits;
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(kGroupThreads), 0, resolve_stream(stream), offsets, order, where, ids, T * top, E, bits);
    return last_launch_status();
}

int ntk_clipped_glu(float* a, const float* gu, int rows, int ff, float limit, float alpha, void* stream) {
    return ntk_glu(a, gu, rows, ff, limit, alpha, 1.0f, stream);
}

int ntk_glu(float* a, const float* gu, int rows, int ff, float limit, float alpha, float up_offset, void* stream) {
    return ntk_glu_rows(a, ff, gu, 2 * ff, rows, ff, limit, alpha, 0.0f, up_offset, stream);
}

int ntk_glu_cubic(float* a, const float* gu, int ldgu, int rows, int ff, float limit, float alpha, float cubic, float up_offset, void* stream) {
    return ntk_glu_rows(a, ff, gu, ldgu, rows, ff, limit, alpha, cubic, up_offset, stream);
}

int ntk_glu_rows(float* a, int lda, const float* gu, int ldgu, int rows, int ff, float limit, float alpha, float cubic, float up_offset, void* stream) {
    if (!a || !gu) return NTK_E_NULL;
    if (rows < 0 || ff <= 0 || ldgu < 2 * ff || lda < ff) return NTK_E_SHAPE;
    if (rows == 0) return NTK_OK;
    const bool vec = ff % 4 == 0 && lda % 4 == 0 && ldgu % 4 == 0 && !(((uintptr_t)a | (uintptr_t)gu) & 15);
    if (vec) hipLaunchKernelGGL(clipped_glu_kernel<4>, dim3((ff / 4 + 255) / 256, rows), dim3(256), 0, resolve_stream(stream), a, lda, gu, ldgu, ff, limit, alpha, cubic, up_offset);
    else hipLaunchKernelGGL(clipped_glu_kernel<1>, dim3((ff + 255) / 256, rows), dim3(256), 0, resolve_stream(stream), a, lda, gu, ldgu, ff, limit, alpha, cubic, up_offset);
    return last_launch_status();
}

int ntk_moe_combine(float* x, const float* mix, const float* d, const int* where, const float* wts, const float* shared, const float* sgate, int T, int top,
                    int n, void* stream) {
    if (!x || !d || !where || !wts || (shared && !sgate)) return NTK_E_NULL;
    if (T < 0 || top <= 0 || n <= 0) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    return launch_combine<true>(x, mix, d, where, wts, shared, sgate, T, top, n, nullptr, 0, nullptr, 0, resolve_stream(stream));
}

int ntk_moe_sum(float* out, const float* d, const int* where, const float* wts, const float* shared, const float* sgate, int T, int top, int n, void* stream) {
    if (!where) return NTK_E_NULL;
    return ntk_moe_sum_ex(out, d, where, nullptr, 0, nullptr, 0, wts, shared, sgate, T, top, n, stream);
}

int ntk_moe_sum_ex(float* out, const float* d, const int* where, const int* ids, int n_experts, const float* h, int ldh, const float* wts, const float* shared,
                   const float* sgate, int T, int top, int n, void* stream) {
    if (!out || !d || !wts || (ids && !h)) return NTK_E_NULL;
    if (T < 0 || top <= 0 || n <= 0 || (ids && ldh < n)) return NTK_E_SHAPE;
    if (T == 0) return NTK_OK;
    return launch_combine<false>(out, nullptr, d, where, wts, shared, sgate, T, top, n, ids, n_experts, h, ldh, resolve_stream(stream));
}
