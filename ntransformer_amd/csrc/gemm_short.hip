// gemm_short.hip -- a short prompt's projections (2 .. 16 tokens) through K-quant tensors of the decode repack (gemv_rp.hip: layout), over planes of a scale per token and 256 columns.
//
// What bounds such a launch is the weights' way from memory, and what kept gemm_f16.hip's form from it was the way inside the CU: tensor -> registers -> an image in LDS -> registers, the planes out of LDS
// once per 16 rows, 22 vector instructions a step.  Here a wave keeps ONE unit of 256 columns: its planes lie in registers for the whole launch (16 KB a wave), a lane's 16 bytes of the tensor are operand
// bytes as they arrive, and LDS holds nothing but the sums of the workgroup's units.  13 vector instructions a step (Q4_K):
//   * Q4_K, Q5_K: a lane's columns are 16 neighbours, so one product spans sub-blocks of different scale and the scale goes into the weight: q sc <= 31 x 63 is exact in FP16.  1024 + q is one v_and_or
//     (mask, exponent), (1024 + q) sc - 1024 sc one v_pk_fma with an exact result; a high nibble stays where it is, at sixteen times its value.
//   * Q6_K: (q - 32) sc takes 13 bits.  Four lane groups exchange dwords (v_permlane32_swap, v_permlane16_swap), after which a product lies within sixteen columns and its sum takes the scale.
// The integers are given to the matrix cores as normal numbers: as FP16 subnormals (q 2^-24, no instruction at all) products come out exact, but their sums are aligned by the nominal exponent and lose
// up to ten bits (root mean square of the error 1.45e-7 -> 2.5e-7, beside towering channels 2.3e-7 -> 1.8e-6).  A product of 22 bits an entry is rounded as it is summed, which the other form's (weights
// of 4 or 5 bits) is not, so the rest of the way is short: no product's sum is the start of another (but for the second pieces), a unit's and a slice's sums are added up as trees (Q6_K, whose products
// are exact: a chain of eight a half of a unit, units in order).  Root mean square of the error over the products' size, this form / the other, 16 x 28672 x 4096: Q4_K 1.393e-7 / 1.476e-7, with eight
// channels a hundred times the others' (24 choices of them) 1.772 / 1.808; Q5_K 1.425 / 1.501, 1.732 / 1.804; Q6_K 1.039 / 1.122, 1.071 / 1.162.  With products in chains of two and units in order it was 2 % more
// beside such channels (and a launch of 57344 x 8192 in Q5_K took 47.0 us instead of 48.5).
// us, 28672 x 4096 in Q4_K: without the planes' way 1.2 less, without any product 3.6 less; three items under way 0.5 .. 1 ahead of four, three ahead of six (4 us).
#include "gemm_short.hip.h"
#include <algorithm>
#include <cstdlib>

namespace ntk {

template <int DT> struct Sp;       // bytes of an item (16 rows x 256 columns): one of its two nibble planes with its fifth / sixth bits, its rows' records; bytes of those bits a lane has per plane
template <> struct Sp<NTK_DT_Q4_K> { static constexpr int S1 = 1024, S2 = 320, HI = 0; };
template <> struct Sp<NTK_DT_Q5_K> { static constexpr int S1 = 1280, S2 = 320, HI = 4; };
template <> struct Sp<NTK_DT_Q6_K> { static constexpr int S1 = 1536, S2 = 288, HI = 8; };

constexpr int SS_WAVES = 8, SS_AHEAD = 3;      // waves of a workgroup; items of a wave under way, and tiles between two barriers

template <int DT> struct SsItem { u32x4 q[2]; uint32_t hi[2 * (Sp<DT>::HI / 4) + (Sp<DT>::HI ? 0 : 1)]; u32x4 rec; uint32_t dd; };

// a: FP16 pair 1024 + n (an integer n < 1024 in the mantissa's place); n s = (1024 + n) s - 1024 s, exact where n s is
__device__ __forceinline__ uint32_t ss_mul(uint32_t a, f16x2 s, f16x2 less) { return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, a), s, less)); }
__device__ __forceinline__ f16x8 ss_op(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return __builtin_bit_cast(f16x8, u32x4{a, b, c, d}); }

// exchange of four dwords among the four groups of sixteen lanes: r[k] of group g -> r[g] of group k
__device__ __forceinline__ void ss_turn(uint32_t (&r)[4]) {
    auto a = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    r[0] = c[0]; r[1] = c[1]; r[2] = d[0]; r[3] = d[1];
}

typedef f32x4 SsSums[SS_AHEAD * SS_WAVES][64];
// the sums of a slice's units (a tree: all requested at once; behind the last: zeros)
template <int N>
__device__ __forceinline__ f32x4 ss_tree(const f32x4 (*of)[64], int n, int lane) {
    f32x4 v[N];
#pragma unroll
    for (int w = 0; w < N; ++w) v[w] = of[min(w, n - 1)][lane];
#pragma unroll
    for (int w = 1; w < N; ++w)
        if (w >= n) v[w] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int step = 1; step < N; step *= 2)
#pragma unroll
        for (int w = 0; w + step < N; w += 2 * step) v[w] += v[w + step];
    return v[0];
}
template <bool TREE>
__device__ __forceinline__ f32x4 ss_units(const f32x4 (*of)[64], int n, int lane) {
    if constexpr (TREE) return n > 4 ? ss_tree<8>(of, n, lane) : n > 2 ? ss_tree<4>(of, n, lane) : ss_tree<2>(of, n, lane);
    f32x4 y = of[0][lane];
    for (int w = 1; w < n; ++w) y += of[w][lane];
    return y;
}

// Workgroup (x, slice): eight waves, wave = (row group wave / ups, unit slice * ups + wave % ups of 256 columns), tiles (x + k wgx) * groups + row group for k = 0, 1, ...
template <int DT>
__device__ __forceinline__ void short_stream(const ShortStreamParams& p, const int bx, const int slice, const int wgx, const int slices, SsSums (&sums)[2]) {
    using R = Sp<DT>;
    constexpr bool FOLD = DT != NTK_DT_Q6_K;
    constexpr int ITEM1 = 2 * R::S1;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), i = lane & 15, g = lane >> 4;
    const int grp = wave / p.ups, first = slice * p.ups, here = min(p.ups, p.units - first);         // the slice's units
    const int u = min(first + wave % p.ups, p.units - 1);
    const bool works = grp < p.groups && wave % p.ups < here;
    const int stride = wgx * p.groups, turns = (p.tiles + stride - 1) / stride, tile0 = bx * p.groups + grp;

    // 1 / rms of the lane's tokens (4 g + e): the parts of the rows' sums of squares are asked for first, added up behind the other requests
    f32x4 part[8];
    if (p.ssq)
#pragma unroll
        for (int k = 0; k < 8; ++k) part[k] = *reinterpret_cast<const f32x4*>(p.ssq + min(k, p.nssq - 1) * GB_SHORT + 4 * g);
    __builtin_amdgcn_sched_barrier(0);
    // ---- the unit's planes, into registers for good ----
    u32x4 x[GB_PLANES][8];
    {
        const uint8_t* base = p.xb + (size_t)u * 8 * GB_STEP_BYTES;
#pragma unroll
        for (int pl = 0; pl < GB_PLANES; ++pl)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                if constexpr (FOLD) {      // product m = (s, h, t) = (m / 4, m / 2 % 2, m % 2): lane group g multiplies columns 128 s + 64 h + 16 g + 8 t + 0 .. 7
                    const uint8_t* rec = base + (size_t)((m >> 1) * 2 + (g >> 1)) * GB_STEP_BYTES + pl * 4 * GB_PIECE + 8 * (g & 1) + (i + 32 * (m & 1)) * 16;
                    const uint64_t a = *reinterpret_cast<const uint64_t*>(rec), b = *reinterpret_cast<const uint64_t*>(rec + 256);
                    x[pl][m] = u32x4{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
                } else x[pl][m] = *reinterpret_cast<const u32x4*>(base + (size_t)m * GB_STEP_BYTES + pl * 4 * GB_PIECE + lane * 16);
            }
    }
    uint64_t sm[GB_PLANES];
    if constexpr (FOLD)
#pragma unroll
        for (int pl = 0; pl < GB_PLANES; ++pl)
            sm[pl] = *reinterpret_cast<const uint64_t*>(p.aux + (size_t)u * GB_MIN_UNIT_BYTES + pl * (GB_MIN_UNIT_BYTES / 2) + ((g & 1) * 16 + i) * 8);
    const f32x4 ginv = *reinterpret_cast<const f32x4*>(p.group_inv + (size_t)u * GB_SHORT + 4 * g);
    __builtin_amdgcn_sched_barrier(0);

    // ---- the tensor's items, SS_AHEAD under way ----
    SsItem<DT> ring[SS_AHEAD];
    auto request = [&](SsItem<DT>& it, int k) {
        const int tile = min(tile0 + k * stride, p.tiles - 1);
        const uint32_t on = k < turns ? ~0u : 0u;                    // (past the last: every lane asks for the same bytes -- straight-line code, exact waits, no traffic)
        int sg = 0;
        if (p.nseg > 1 && tile >= p.seg[1].tile0) sg = 1;
        if (p.nseg > 2 && tile >= p.seg[2].tile0) sg = 2;
        const uint32_t item = (uint32_t)(tile - p.seg[sg].tile0) * (uint32_t)p.units + (uint32_t)u;
        const uint8_t* q = p.seg[sg].W + (size_t)item * ITEM1;
        const uint8_t* rec = p.seg[sg].W + p.seg[sg].p2_off + (size_t)item * R::S2;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            it.q[s] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(q + s * R::S1 + (lane * 16 & on)));
            if constexpr (R::HI == 4) it.hi[s] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(q + s * R::S1 + 1024 + (lane * 4 & on)));
            if constexpr (R::HI == 8) {
                const uint64_t v = __builtin_nontemporal_load(reinterpret_cast<const uint64_t*>(q + s * R::S1 + 1024 + (lane * 8 & on)));
                it.hi[2 * s] = (uint32_t)v; it.hi[2 * s + 1] = (uint32_t)(v >> 32);
            }
        }
        it.rec = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(rec + (i * 16 & on)));
        if constexpr (FOLD) it.dd = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(rec + 256 + (i * 4 & on)));
        else it.dd = __builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(rec + 256 + (i * 2 & on)));
    };
    if (works) {
#pragma unroll
        for (int a = 0; a < SS_AHEAD; ++a) { request(ring[a], a); __builtin_amdgcn_sched_barrier(0); }
    }
    f32x4 rms = {1.0f, 1.0f, 1.0f, 1.0f};
    if (p.ssq) {
        f32x4 q = part[0];
#pragma unroll
        for (int k = 1; k < 8; ++k)
            if (k < p.nssq) q += part[k];
        for (int k = 8; k < p.nssq; ++k) q += *reinterpret_cast<const f32x4*>(p.ssq + k * GB_SHORT + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) rms[e] = 1.0f / sqrtf(q[e] / (float)p.in + p.eps);
    }
    if constexpr (FOLD)            // columns (0, 2), (1, 3), ... of a product, as the nibbles of a dword come out of it
#pragma unroll
        for (int pl = 0; pl < GB_PLANES; ++pl)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const u32x4 v = x[pl][m];
                x[pl][m] = u32x4{__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                                 __builtin_amdgcn_perm(v.w, v.z, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u)};
            }
    // (everything but the items has landed here: a first use inside the loop would wait for the items too)
#pragma unroll
    for (int pl = 0; pl < GB_PLANES; ++pl) {
#pragma unroll
        for (int m = 0; m < 8; ++m) asm volatile("" : "+v"(x[pl][m]));
        if constexpr (FOLD) asm volatile("" : "+v"(sm[pl]));
    }
    asm volatile("" :: "v"(ginv), "v"(rms));
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t k6400 = 0x64006400u, mlo = 0x000F000Fu, mhi = 0x00F000F0u;      // (one instruction for mask and exponent: its operands in registers)
    asm volatile("" : "+v"(k6400));
    asm volatile("" : "+s"(mlo), "+s"(mhi));
    auto multiply = [&](const SsItem<DT>& it) {
        f32x4 y;
        if constexpr (FOLD) {
            f32x4 acc[2][2][2], low0 = zero, low1 = zero;        // [s][h][t] of the first pieces
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                // the sub-blocks' scales of this lane's columns as FP16, (low nibbles, high nibbles): 1024 + sc, less 1024; a high nibble stands at sixteen times its value, and so do those products
                const uint32_t w = ((s ? it.rec.y : it.rec.x) >> (8 * (g >> 1))) & 0x00FF00FFu;
                const f16x2 sc = __builtin_bit_cast(f16x2, w | 0x64006400u) + f16x2{(_Float16)-1024.0f, (_Float16)-1024.0f};
                const f16x2 less = sc * f16x2{(_Float16)-1024.0f, (_Float16)-1024.0f}, s0 = {sc.x, sc.x}, s1 = {sc.y, sc.y}, n0 = {less.x, less.x}, n1 = {less.y, less.y};
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    uint32_t lo[4], hi[4];
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const int v = 2 * t + c;
                        const uint32_t a = it.q[s][v], b = a >> 8;
                        uint32_t l0 = (a & mlo) | k6400, l1 = (b & mlo) | k6400, h0 = (a & mhi) | k6400, h1 = (b & mhi) | k6400;
                        if constexpr (R::HI == 4) {       // fifth bits of columns 4 v + y: bit 8 y + v (low), 8 y + 4 + v (high)
                            const uint32_t f = it.hi[s] << (4 - v), fy = it.hi[s] >> (4 + v);
                            l0 |= f & 0x00100010u; l1 |= fy & 0x00100010u; h0 |= f & 0x01000100u; h1 |= fy & 0x01000100u;
                        }
                        lo[2 * c] = ss_mul(l0, s0, n0); lo[2 * c + 1] = ss_mul(l1, s0, n0);
                        hi[2 * c] = ss_mul(h0, s1, n1); hi[2 * c + 1] = ss_mul(h1, s1, n1);
                    }
                    const f16x8 wl = ss_op(lo[0], lo[1], lo[2], lo[3]), wh = ss_op(hi[0], hi[1], hi[2], hi[3]);
                    acc[s][0][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[0][4 * s + t]), wl, zero, 0, 0, 0);
                    low0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[1][4 * s + t]), wl, low0, 0, 0, 0);
                    acc[s][1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[0][4 * s + 2 + t]), wh, zero, 0, 0, 0);
                    low1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x[1][4 * s + 2 + t]), wh, low1, 0, 0, 0);
                }
            }
            // the minima: m_0 .. m_3 in lane group 0, m_4 .. m_7 in group 1
            const uint32_t w = (it.rec.z & (g == 0 ? ~0u : 0u)) | (it.rec.w & (g == 1 ? ~0u : 0u));
            const f16x2 k1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
            auto whole = [&](uint32_t v) { return __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, v) + k1024)); };
            const f16x8 mb = ss_op(whole(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)), whole(__builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)), 0u, 0u);
            f32x4 mn = zero;
#pragma unroll
            for (int pl = 0; pl < GB_PLANES; ++pl) {
                const uint32_t a = (uint32_t)sm[pl], b = (uint32_t)(sm[pl] >> 32);
                mn = __builtin_amdgcn_mfma_f32_16x16x32_f16(ss_op(a, b, a, b), mb, mn, 0, 0, 0);
            }
            const float d = h2f((uint16_t)(it.dd & 0xFFFFu)), dm = h2f((uint16_t)(it.dd >> 16)) * -64.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                auto first = [&](int h) { return (acc[0][h][0][e] + acc[0][h][1][e]) + (acc[1][h][0][e] + acc[1][h][1][e]); };
                y[e] = fmaf(d, fmaf(0.0625f, first(1) + low1[e], first(0) + low0[e]), dm * mn[e]);
            }
        } else {
            f32x4 half[2] = {zero, zero};                 // a chain of eight a half of the unit
            const float d = h2f((uint16_t)it.dd);
            const f16x2 off = {(_Float16)-1056.0f, (_Float16)-1056.0f};
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t r[4];
                    const uint32_t f = it.hi[2 * s + h];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {         // whole six-bit values of columns 4 v + y: bits 8 y + 2 v (+ 1) of f above the nibbles
                        const uint32_t up = v < 2 ? f << (4 - 2 * v) : v == 2 ? f : f >> 2;
                        r[v] = ((it.q[s][v] >> (4 * h)) & 0x0F0F0F0Fu) | (up & 0x30303030u);
                    }
                    ss_turn(r);                           // columns 4 g + y of the sixteen columns k
                    const uint32_t scw = s ? (h ? it.rec.w : it.rec.z) : (h ? it.rec.y : it.rec.x);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, r[k], 0x04010400u)) + off, b = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, r[k], 0x04030402u)) + off;
                        const f16x4 w = {a.x, a.y, b.x, b.y};
                        f32x4 c = zero;
#pragma unroll
                        for (int pl = 0; pl < GB_PLANES; ++pl) {
                            const u32x4 xv = x[pl][4 * s + 2 * h + (k >> 1)];
                            const f16x4 xk = __builtin_bit_cast(f16x4, k & 1 ? (uint64_t)xv.z | ((uint64_t)xv.w << 32) : (uint64_t)xv.x | ((uint64_t)xv.y << 32));
                            c = __builtin_amdgcn_mfma_f32_16x16x16f16(xk, w, c, 0, 0, 0);
                        }
                        const float sc = d * (float)(int)(int8_t)(scw >> (8 * k));
#pragma unroll
                        for (int e = 0; e < 4; ++e) half[s][e] = fmaf(sc, c[e], half[s][e]);
                    }
                }
            y = half[0] + half[1];
        }
        return y * ginv;
    };
    for (int k0 = 0; k0 < turns; k0 += SS_AHEAD) {
        SsSums& buf = sums[(k0 / SS_AHEAD) & 1];
        if (works)
#pragma unroll
            for (int a = 0; a < SS_AHEAD; ++a) {
                if (k0 + a < turns) buf[a * SS_WAVES + wave][lane] = multiply(ring[a]);       // (uniform; past the last tile nothing reads it)
                __builtin_amdgcn_sched_barrier(0);
                request(ring[a], k0 + a + SS_AHEAD);
                __builtin_amdgcn_sched_barrier(0);
            }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");       // (the requests stay under way; the other buffer's sums were read in front of this)
        for (int l = wave; l < SS_AHEAD * p.groups; l += SS_WAVES) {
            const int a = l / p.groups, gr = l - a * p.groups, tile = (bx + (k0 + a) * wgx) * p.groups + gr;
            if (k0 + a >= turns || tile >= p.tiles) continue;
            const f32x4 y = ss_units<FOLD>(&buf[a * SS_WAVES + gr * p.ups], here, lane);
            int sg = 0;
            if (p.nseg > 1 && tile >= p.seg[1].tile0) sg = 1;
            if (p.nseg > 2 && tile >= p.seg[2].tile0) sg = 2;
            const int r = (tile - p.seg[sg].tile0) * 16 + i, out = p.seg[sg].out;
            if (r >= out) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 4 * g + e;
                if (t >= p.T) continue;
                const float v = y[e] * rms[e];
                if (slices > 1) p.seg[sg].part[((size_t)slice * p.T + t) * out + r] = v;
                else { const size_t at = (size_t)t * out + r; p.seg[sg].Y[at] = p.resid ? v + p.resid[at] : v; }
            }
        }
    }
}

template <int DT>
__global__ __launch_bounds__(64 * SS_WAVES, 2) void short_stream_kernel(const ShortStreamParams p) {
    __shared__ __attribute__((aligned(16))) SsSums sums[2];
    short_stream<DT>(p, blockIdx.x, blockIdx.y, gridDim.x, gridDim.y, sums);
}

// matrices of two formats over the same planes (a K-quant mix keeps more bits of some): a.wgx columns of workgroups have the first format's, the others the second's
template <int DA, int DB>
__global__ __launch_bounds__(64 * SS_WAVES, 2) void short_stream_two_kernel(const ShortStreamParams a, const ShortStreamParams b, const int wgx) {
    __shared__ __attribute__((aligned(16))) SsSums sums[2];
    if ((int)blockIdx.x < wgx) short_stream<DA>(a, blockIdx.x, blockIdx.y, wgx, gridDim.y, sums);
    else short_stream<DB>(b, (int)blockIdx.x - wgx, blockIdx.y, (int)gridDim.x - wgx, gridDim.y, sums);
}

// Turns (tiles a wave takes) decide: the chip's 256 workgroups are there at once.  us of a launch, this form / the one with its planes in LDS, 16 tokens: gate | up of 28672 x 4096 (14 turns, two slices) Q4_K
// 21.0 / 26.4, Q5_K 25.0 / 29.5, Q6_K 28.0 / 34.8; 57344 x 8192 (56 turns) 60 / 83, 93 / 97, 95 / 117; 8192 x 28672 (29) 36 / 42, 50 / 50, 53 / 60; Q | K | V of 4096 columns (3) 9.6 / 10.6, 10.8 / 11.9, 11.6 / 12.3;
// behind it: 4096 x 4096 (2) 8.5 / 7.2, 9.3 / 8.3, 9.8 / 8.5, 4096 x 14336 (8) 14.6 / 13.2, 17.3 / 14.8, 18.7 / 17.0, 1024 x 4096 (1) 9 / 6.9 -- a wave reads 16 KB of planes before its first
// product.  `other`: steps of 32 columns a wave of that form takes one after the other.
static float turn_us(int dt) { return dt == NTK_DT_Q4_K ? 1.03f : dt == NTK_DT_Q5_K ? 1.3f : 1.54f; }
ShortStreamPlan short_stream_plan(int dt, int units, int tiles, int most, int other) {
    ShortStreamPlan b;
    const float turn = turn_us(dt), step = dt == NTK_DT_Q4_K ? 0.15f : dt == NTK_DT_Q5_K ? 0.17f : 0.22f;
    float best = 5.0f + step * (float)other;
    for (int ups = 1; ups <= std::min(units, SS_WAVES); ++ups) {
        const int n = (units + ups - 1) / ups, groups = SS_WAVES / ups;
        if (n > most || n > 256 || (units + n - 1) / n != ups) continue;      // (ups: the units evenly over the slices)
        const int wgx = std::max(1, std::min((tiles + groups - 1) / groups, 256 / n)), turns = (tiles + wgx * groups - 1) / (wgx * groups);
        const float us = 6.3f + turn * (float)turns + 0.1f * (float)n;
        if (us < best) { best = us; b.n = n; b.ups = ups; b.groups = groups; b.wgx = wgx; }
    }
    b.us = best;
    return b;
}

// Two formats in one launch: the chip's workgroups shared so that the one that ends last ends as early as can be.  Against two launches (apart: their estimates) what is saved is mostly the second
// one's way to its first product: us, 16 tokens, 5120 rows in Q4_K and 1024 in Q6_K, 4096 columns: 10.4 + 6.8 -> 12.0; short prompts through eight 8B-shaped layers in Q4_K_M 673 -> 645 (2 tokens),
// 735 -> 709 (16), eight 70B-shaped ones (Q4_K and Q5_K or Q6_K) 1389 -> 1347, 1534 -> 1469.
bool short_stream_plan_two(int da, int db, int units, int tiles_a, int tiles_b, int most, float apart, ShortStreamPlan* a, ShortStreamPlan* b) {
    float best = apart;
    bool found = false;
    for (int ups = 1; ups <= std::min(units, SS_WAVES); ++ups) {
        const int n = (units + ups - 1) / ups, groups = SS_WAVES / ups;
        if (n > most || n > 128 || (units + n - 1) / n != ups) continue;
        const int room = 256 / n;
        for (int wa = 1; wa < room; ++wa) {
            const int wb = room - wa, ta = (tiles_a + wa * groups - 1) / (wa * groups), tb = (tiles_b + wb * groups - 1) / (wb * groups);
            const float us = 6.8f + std::max(turn_us(da) * (float)ta, turn_us(db) * (float)tb) + 0.1f * (float)n;
            if (us >= best) continue;
            best = us;
            found = true;
            *a = *b = ShortStreamPlan{n, ups, groups, std::min(wa, (tiles_a + groups - 1) / groups), us};
            b->wgx = std::min(wb, (tiles_b + groups - 1) / groups);
        }
    }
    return found;
}

int short_stream_launch(int dt, const ShortStreamParams& p, const ShortStreamPlan& plan, hipStream_t st) {
    const dim3 grid(plan.wgx, plan.n), block(64 * SS_WAVES);
    switch (dt) {
        case NTK_DT_Q4_K: hipLaunchKernelGGL(short_stream_kernel<NTK_DT_Q4_K>, grid, block, 0, st, p); break;
        case NTK_DT_Q5_K: hipLaunchKernelGGL(short_stream_kernel<NTK_DT_Q5_K>, grid, block, 0, st, p); break;
        case NTK_DT_Q6_K: hipLaunchKernelGGL(short_stream_kernel<NTK_DT_Q6_K>, grid, block, 0, st, p); break;
        default: return NTK_E_DTYPE;
    }
    return last_launch_status();
}

int short_stream_launch_two(int da, int db, const ShortStreamParams& a, const ShortStreamParams& b, const ShortStreamPlan& pa, const ShortStreamPlan& pb, hipStream_t st) {
    const dim3 grid(pa.wgx + pb.wgx, pa.n), block(64 * SS_WAVES);
    if (da == NTK_DT_Q4_K && db == NTK_DT_Q5_K) hipLaunchKernelGGL((short_stream_two_kernel<NTK_DT_Q4_K, NTK_DT_Q5_K>), grid, block, 0, st, a, b, pa.wgx);
    else if (da == NTK_DT_Q4_K && db == NTK_DT_Q6_K) hipLaunchKernelGGL((short_stream_two_kernel<NTK_DT_Q4_K, NTK_DT_Q6_K>), grid, block, 0, st, a, b, pa.wgx);
    else if (da == NTK_DT_Q6_K && db == NTK_DT_Q5_K) hipLaunchKernelGGL((short_stream_two_kernel<NTK_DT_Q6_K, NTK_DT_Q5_K>), grid, block, 0, st, a, b, pa.wgx);
    else return NTK_E_DTYPE;
    return last_launch_status();
}

}  // namespace ntk
