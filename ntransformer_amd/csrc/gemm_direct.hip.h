// gemm_direct.hip.h -- tiled products Y[r][n] = sum_k X[r][k] W[n][k] whose operands lie in memory as the matrix cores take them.
//
// The form of gemm_tile.hip.h converts activations in every workgroup, on their way through registers into LDS: each of a product's up to 117 column tiles reads 32-bit
// activations and rounds them again, and with the operands' way through registers a workgroup of eight waves is left with wave tiles of 32 x 64, for which LDS has to
// deliver 192 bytes a cycle and CU at the matrix cores' full rate, where it has 128.  Here the activations were rounded (or cut into pieces) once, by the launch that wrote them or
// by one in front of the product; both operands go from memory straight into LDS (global_load_lds, 16 bytes a lane), STAGES chunks of 128 bytes a row deep, and a wave of the large forms owns 64 x 64 or
// 64 x 128 (96 .. 128 bytes).  What bounds the large ones is the matrix cores: a 64-input chunk of 256 x 256
// tiles on every CU is 2.15 GFLOP, 0.86 us at their dense peak and 1.77 us at the rate of a large library product (1216 TF/s); whole products of 1024 .. 2048 rows run at 930 .. 1010 TF/s.
// (The 1.45 us a chunk in plan_direct_bf16 is a constant fitted together with `over`, the latency of the first chunks and the results on their way out, which is what bounds products
// below a few tiles a CU: no measured rate.)  Consecutive tiles of an XCD share their weights.
// Measured (us, weights from memory; the form of gemm_tile.hip.h with its best tile and pieces): bf16 1024 x 14976 x 2048 142 -> 62 (1010 TF/s), 1024 x 2048 x 7488 63 -> 43,
// 1024 x 6240 x 2048 58 -> 37, 1024 x 2048 x 2048 26 -> 16.5, 40 x 14976 x 2048 22 -> 17, 6144 rows in 32 groups of 2816 x 2048 227 -> 133, of 2048 x 1408 116 -> 72.
// One chain of matrix instructions over the inputs as there: the same bits where K is not cut.
#pragma once
#include "gemm_tile.hip.h"

namespace ntk {

struct DirectArgs {
    TileArgs t;                                     // X unused
    const void* X16; uint32_t x_row; long long plane;      // activations as the matrix cores take them, rows of x_row bytes; PIECES planes, `plane` bytes apart
    uint16_t* Y16; int ldy16; int glu_ff;           // bfloat16 results in the place of t.Y (or NULL); gated units: [r][f] of the weight rows f behind gate_at and up_at bytes of W
    uint32_t gate_at, up_at;
    float limit, alpha, up_offset, cubic;
    int tile_rows;                                  // EVEN forms: rows of a tile, whole pieces of sixteen
    // several matrices side by side over the same activations (n_seg > 1, no groups, nothing accumulated): the column tiles of one after those of the other, their pieces' columns too
    int n_seg; const void* segW[3]; float* segY[3]; int seg_out[3], seg_tile[3];
};
enum { kGluNone = 0, kGluClipped = 1, kGluSilu = 2 };       // kGluSilu: silu(gate) * up as F32, as a launch of its own forms it
template <typename T> __device__ __forceinline__ T seg_pick(const T (&v)[3], int i) { return i == 0 ? v[0] : i == 1 ? v[1] : v[2]; }

// N requests of 16 bytes a lane: lane l's land at lds + i * step + 16 l.  The compiler does not count them (M0 is the compiler's: saved and restored)
template <int STEP>
__device__ __forceinline__ void direct_load4(uint32_t lds, const void* base, uint32_t o0, uint32_t o1, uint32_t o2, uint32_t o3) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %1\n\t"
                 "s_add_u32 m0, m0, %7\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %1\n\t"
                 "s_add_u32 m0, m0, %7\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %1\n\t"
                 "s_add_u32 m0, m0, %7\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %6, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(o0), "v"(o1), "v"(o2), "v"(o3), "i"(STEP) : "memory", "scc");
}
__device__ __forceinline__ void direct_load1(uint32_t lds, const void* base, uint32_t o0) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(o0) : "memory");
}
template <int STEP>
__device__ __forceinline__ void direct_load2(uint32_t lds, const void* base, uint32_t o0, uint32_t o1) {
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %1\n\t"
                 "s_add_u32 m0, m0, %5\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %1\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "s"(base), "s"(lds), "v"(o0), "v"(o1), "i"(STEP) : "memory", "scc");
}
template <int N, int STEP>
__device__ __forceinline__ void direct_load(uint32_t lds, const void* base, const uint32_t (&o)[N]) {
    constexpr int F = N / 4 * 4;
#pragma unroll
    for (int i = 0; i < F; i += 4) direct_load4<STEP>(lds + i * STEP, base, o[i], o[i + 1], o[i + 2], o[i + 3]);
    if constexpr (N % 4 >= 2) direct_load2<STEP>(lds + F * STEP, base, o[F], o[F + 1]);
    if constexpr (N % 2) direct_load1(lds + (N - 1) * STEP, base, o[N - 1]);
}
template <int V> __device__ __forceinline__ void direct_wait() {   // all but the newest V requests have landed, this wave's LDS reads are done, and so everywhere in the workgroup
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "i"(V) : "memory");
}

// one-dimensional grid over (row tiles, column tiles, splits), row tiles first; rows of X and W are whole multiples of 128 bytes
template <class P, int TM, int TN, int WM, int WN, int STAGES, int GLU, int MINW>
__global__ __launch_bounds__(64 * WM * WN, MINW) void gemm_direct_kernel(const DirectArgs d, const int row_tiles, const int col_tiles) {
    const TileArgs& a = d.t;
    constexpr int CB = 128, ES = sizeof(typename P::WT), BK = CB / ES, PIECES = P::PIECES, NW = WM * WN, WTM = TM / WM, WTN = TN / WN, MI = WTM / 16, NJ = WTN / 16;
    constexpr int NX = TM / (8 * NW), NWL = TN / (8 * NW), LPS = NX * PIECES + NWL;      // requests of a wave: X per plane, W; per chunk
    constexpr int XB = TM * CB, STAGE = (PIECES * TM + TN) * CB;
    // the rows go evenly over the tiles (never in groups): two pieces an activation leave the matrix cores and LDS both full, so that rows a tile does not have count.  200 rows 112 -> 107 us, 130 111 -> 92
    // (28672 x 4096), 130 of 4096 x 14336 in eight pieces 54 -> 47.  Not smaller tiles (64 x 128: 51 -> 54, what a step asks each time) and not bfloat16, which waits for its weights then (even tiles of
    // 1024 rows in 32 groups of 2816 x 2048: no gain)
    constexpr bool EVEN = PIECES > 1 && TM >= 128;
    static_assert(TM % (8 * NW) == 0 && TN % (8 * NW) == 0, "whole requests");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * STAGE];
    // consecutive workgroups go to the eight XCDs in turn: each takes a contiguous range of tiles, so that the row tiles of a column share its weights in one L2
    const int n_wg = gridDim.x, xcd = blockIdx.x & 7, per = n_wg >> 3, rem = n_wg & 7;
    int id = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
    const int rt = id % row_tiles;
    id /= row_tiles;
    int ct = id % col_tiles;
    const int split = id / col_tiles;
    const void* Wp = a.W;
    float* Yp = a.Y;
    int n_cols = GLU ? d.glu_ff : a.N, ldy = a.ldy, part_col = 0;
    if (!GLU && d.n_seg > 1) {
        const int sg = (ct >= d.seg_tile[1] ? 1 : 0) + (d.n_seg > 2 && ct >= d.seg_tile[2] ? 1 : 0);
        ct -= sg ? seg_pick(d.seg_tile, sg) : 0;
        Wp = seg_pick(d.segW, sg); Yp = seg_pick(d.segY, sg); n_cols = ldy = seg_pick(d.seg_out, sg);
        part_col = (sg > 0 ? d.seg_out[0] : 0) + (sg > 1 ? d.seg_out[1] : 0);
    }
    int g = 0, row_base = rt * (EVEN ? d.tile_rows : TM), r1 = EVEN ? min(a.T, row_base + d.tile_rows) : a.T;
    if (a.offsets) { if (!group_tile(a.offsets, a.G, rt, TM, g, row_base, r1)) return; }
    const int n_base = ct * (GLU ? TN / 2 : TN);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = EVEN ? wave / WN : wave % WM, wn = EVEN ? wave % WN : wave / WM;
    const int k_begin = split * a.k_per_split, k_end = min(a.K, k_begin + a.k_per_split), n_chunks = (k_end - k_begin) / BK;
    // a request brings eight rows of 128 bytes; the 16-byte pieces of row r are stored in the order piece ^ (r & 7)
    uint32_t xo[NX], wo[NWL];
    const uint32_t row_bytes = (uint32_t)a.K * ES;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int row = (i * NW + wave) * 8 + (lane >> 3), r = min(row_base + row, r1 - 1), src = a.rows ? a.rows[r] / a.row_div : r;
        xo[i] = (uint32_t)src * d.x_row + (uint32_t)(((lane & 7) ^ (row & 7)) * 16);
    }
#pragma unroll
    for (int i = 0; i < NWL; ++i) {
        const int row = (i * NW + wave) * 8 + (lane >> 3);
        if constexpr (GLU != kGluNone) {            // a wave's columns: as many gates as the up rows of the same outputs behind them
            const int n = min(n_base + (row / WTN) * (WTN / 2) + row % (WTN / 2), n_cols - 1);
            wo[i] = (uint32_t)n * row_bytes + (row % WTN >= WTN / 2 ? d.up_at : d.gate_at);
        } else wo[i] = (uint32_t)(min(n_base + row, n_cols - 1) - n_base) * row_bytes;
        wo[i] += (uint32_t)(((lane & 7) ^ (row & 7)) * 16);
    }
    const char* xb = (const char*)d.X16 + (long long)k_begin * ES;
    const char* wb = (const char*)Wp + ((long long)g * a.wstride + (GLU ? 0 : (long long)n_base * a.K) + k_begin) * ES;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    const uint32_t mine = lds0 + wave * 1024;
    auto request = [&](int chunk, int slot) {
        const uint32_t at = mine + slot * STAGE;
        const long long off = (long long)chunk * CB;
#pragma unroll
        for (int q = 0; q < PIECES; ++q) direct_load<NX, NW * 1024>(at + q * XB, xb + q * d.plane + off, xo);
        direct_load<NWL, NW * 1024>(at + PIECES * XB, wb + off, wo);
    };
    floatx4_t acc[MI][NJ];
    constexpr bool SEP = PIECES > 1;
    floatx4_t low[SEP ? MI : 1][SEP ? NJ : 1];
    constexpr int RUN_CHUNKS = P::RUN / BK;
    floatx4_t total[RUN_CHUNKS ? MI : 1][RUN_CHUNKS ? NJ : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            if constexpr (SEP) low[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            if constexpr (RUN_CHUNKS > 0) total[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        }
    auto end_run = [&]() {
        if constexpr (RUN_CHUNKS > 0)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) { total[i][j] += acc[i][j]; acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
    };
    // (uniform) EVEN: the tile's pieces of sixteen rows, shared among the waves of a column (wm differs between the two waves of a SIMD, so that each SIMD has its share of those left out)
    const int pieces16 = (r1 - row_base + 15) / 16, n16 = EVEN ? pieces16 / WM + (wm < pieces16 % WM ? 1 : 0) : MI;
    const int first_row = EVEN ? 16 * (wm * (pieces16 / WM) + min(wm, pieces16 % WM)) : wm * WTM, row_end = EVEN ? min(r1, row_base + first_row + 16 * n16) : r1;
    const bool idle = row_base + first_row >= row_end;    // (uniform) rows past the group's end: nothing to multiply, the matrix cores are a neighbour's
    auto multiply = [&](int slot) {
        const uint8_t* s = lds + slot * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int piece = (((h * 4 + (lane >> 4)) ^ (lane & 7)) * 16) + (lane & 15) * CB;
            uintx4_t wf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j) wf[j] = *reinterpret_cast<const uintx4_t*>(s + PIECES * XB + (wn * WTN + j * 16) * CB + piece);
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                uintx4_t xf[MI];
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    if (EVEN && i && i >= n16) break;
                    xf[i] = *reinterpret_cast<const uintx4_t*>(s + q * XB + (first_row + i * 16) * CB + piece);
                }
#pragma unroll
                for (int c = 0; c < P::STEPS; ++c)          // (neighbouring instructions on different accumulators)
#pragma unroll
                    for (int i = 0; i < MI; ++i) {
                        if (EVEN && i && i >= n16) break;
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            if (SEP && q > 0) low[SEP ? i : 0][SEP ? j : 0] = P::step(xf[i], wf[j], low[SEP ? i : 0][SEP ? j : 0], c);
                            else acc[i][j] = P::step(xf[i], wf[j], acc[i][j], c);
                        }
                    }
            }
        }
    };
#pragma unroll
    for (int c = 0; c < STAGES - 1; ++c) if (c < n_chunks) request(c, c);
    int slot = 0;
    for (int i = 0; i < n_chunks; ++i) {
        const int left = n_chunks - 1 - i;          // chunks behind this one
        if (left >= STAGES - 2) direct_wait<LPS * (STAGES - 2)>();
        else if (STAGES > 3 && left == 1) direct_wait<LPS>();
        else direct_wait<0>();
        if (left >= STAGES - 1) request(i + STAGES - 1, slot == 0 ? STAGES - 1 : slot - 1);
        if (!idle) multiply(slot);
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        if constexpr (RUN_CHUNKS > 0) { if ((i + 1) % RUN_CHUNKS == 0) end_run(); }
    }
    if (idle) return;
    if constexpr (SEP)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] += low[i][j];
    if constexpr (RUN_CHUNKS > 0) {
        end_run();
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = total[i][j];
    }
    // accumulator lane map: row 4 * (lane / 16) + r, column lane % 16
    if constexpr (GLU == kGluSilu) {
        const int col = n_base + wn * (WTN / 2) + (lane & 15), n_left = n_cols - col;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int row = row_base + first_row + i * 16 + (lane >> 4) * 4;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool in = row + r < row_end;
                const float undo = P::SCALED ? half_unscale(a.row_max[min(row + r, a.T - 1)]) : 1.0f;
                float* y = Yp + (long long)(row + r) * ldy + col;
#pragma unroll
                for (int j = 0; j < NJ / 2; ++j)
                    if (in && j * 16 < n_left) {
                        const float gg = acc[i][j][r] * undo;
                        y[j * 16] = gg / (1.0f + expf(-gg)) * (acc[i][NJ / 2 + j][r] * undo);
                    }
            }
        }
        return;
    }
    if constexpr (GLU == kGluClipped) {
        const int col = n_base + wn * (WTN / 2) + (lane & 15), n_left = n_cols - col;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const int row = row_base + first_row + i * 16 + (lane >> 4) * 4;
#pragma unroll
            for (int j = 0; j < NJ / 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < row_end && j * 16 < n_left) {
                        const float gg = fminf(acc[i][j][r], d.limit), uu = fminf(fmaxf(acc[i][NJ / 2 + j][r], -d.limit), d.limit);
                        const float zz = d.cubic != 0.0f ? fmaf(d.cubic * gg * gg, gg, gg) : gg;
                        const float v = gg * (1.0f / (1.0f + expf(-d.alpha * zz))) * (uu + d.up_offset);
                        if (d.Y16) d.Y16[(long long)(row + r) * d.ldy16 + col + j * 16] = (uint16_t)pack_bf16(v, 0.0f);
                        else Yp[(long long)(row + r) * ldy + col + j * 16] = v;
                    }
        }
        return;
    }
    const int col = n_base + wn * WTN + (lane & 15), n_left = n_cols - col;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = row_base + first_row + i * 16 + (lane >> 4) * 4;
        float undo[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (P::SCALED)
#pragma unroll
            for (int r = 0; r < 4; ++r) undo[r] = half_unscale(a.row_max[min(row + r, a.T - 1)]);
        if (a.splits > 1) {
            float* y = a.part + ((long long)split * a.T + row) * a.N + part_col + col;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < row_end && j * 16 < n_left) y[(long long)r * a.N + j * 16] = acc[i][j][r] * undo[r];
            continue;
        }
        float* y = Yp + (long long)row * ldy + col;
        float old[NJ][4] = {};
        if (a.accumulate)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) old[j][r] = row + r < row_end && j * 16 < n_left ? y[(long long)r * ldy + j * 16] : 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (row + r < row_end && j * 16 < n_left) {
                    float v = acc[i][j][r] * undo[r];
                    if (a.accumulate) v += old[j][r];
                    else if (a.act == 1) { const float p = fmaxf(v, 0.0f); v = p * p; }          // NTK_ACT_RELU2
                    if (d.Y16) d.Y16[(long long)(row + r) * d.ldy16 + col + j * 16] = (uint16_t)pack_bf16(v, 0.0f);
                    else y[(long long)r * ldy + j * 16] = v;
                }
    }
}

// ---- which tile, and how many pieces of K.  A tile of a form takes `over` us beside its chunks (first requests, results); n of them on a CU, `resident` at a time, take
// n * busy a chunk, one alone `alone` (latency).  Constants in us, from layer-like shapes of 16 .. 1024 rows (groups: 600 .. 6144), 2048 .. 14976 outputs, 512 .. 7488 inputs with weights
// that come from memory; the estimate is within a sixth there, and the choice within a tenth of the best form but for uneven small groups.  Rows of several groups: tiles
// of a group of the average size, plus half a tile where that is no small part of one.
struct DirectForm { int TM, TN, resident; float alone, busy, over, even; };       // even: the part of a chunk's time that goes with the rows a tile has (rows evenly over the tiles)
// rounds (one matrix): a second estimate has a CU's last tiles, where they are no whole number of `resident` ones, at the pace of a tile alone, and looks at five pieces where six put a second tile
// on a CU.  `us` stays the first estimate's (the lines between these forms and others are drawn with it); the plan is the second one's where that has the same tile in fewer pieces, or is ahead by a
// tenth.  Both plans were measured wherever they differ.  bfloat16, 1080 sizes of 9 .. 2000 rows: the same tile in fewer pieces takes 0.88 of the time on average and never more (150 x 2048 x 2048 in
// five for eight 12.7 -> 10.7), a tenth ahead 0.94 (700 x 4096 x 14336 90 -> 80; 15 of 161 are behind by more than 2 %, half of those where 256 x 256 tiles replace two of 128 x 128 a CU, 9 % there and
// 12 % at most); up to a twentieth ahead it is no better than chance, between the two 23 of 64 are behind, by up to 19 %.  Halves of 32-bit activations, 437 sizes (with their split and the sum):
// 0.93 (2 of 24 behind, by 3 %) and 0.955 (6 of 147, 6 % at most); gated 0.90 (4 of 31, 5 %).  Before, where these plans were the first estimate's: 200 x 6144 x 4096 46.8 -> 39.8 (768 tiles of
// 64 x 128 on 512 places / 240 of 128 x 256 in five pieces), gated bfloat16 1181 x 7488 x 7488 212 -> 172.
static TilePlan plan_direct(const DirectForm* f, int n_forms, int chunk, int rows, int groups, int N, int K, long long scratch_floats, bool rounds = false) {
    static const int counts[] = {1, 2, 3, 4, 5, 6, 8, 12, 16};
    TilePlan best{0, 1, 1e30f}, other = best;
    float best_too = 0.0f;                          // the second estimate of `best`
    const int chunks = (K + chunk - 1) / chunk;
    for (int i = 0; i < n_forms; ++i) {
        const float mean = (float)rows / groups / f[i].TM;
        const float row_tiles = groups > 1 ? groups * (mean < 0.5f ? 1.0f : mean + 0.5f) : (float)((rows + f[i].TM - 1) / f[i].TM);
        const float tiles = row_tiles * ((N + f[i].TN - 1) / f[i].TN);
        for (int s : counts) {
            if (s > 1 && ((long long)s * rows * N > scratch_floats || chunks < 4 * s)) break;
            const int n = (int)((tiles * s + 255.0f) / 256.0f), rest = n % f[i].resident;
            const float full = 1.0f - f[i].even * (1.0f - std::min(1.0f, mean / row_tiles));
            const float each = (float)((chunks + s - 1) / s) * full;
            float beside = f[i].over * ((n + f[i].resident - 1) / f[i].resident);
            if (s > 1) beside += 3.0f + (float)(s + 1) * rows * N * 4.0f / 7e6f;
            const float us = each * (n == 1 ? f[i].alone : n * f[i].busy) + beside;
            const float too = each * (n == 1 ? f[i].alone : (n - rest) * f[i].busy + (rest ? std::max(f[i].alone, rest * f[i].busy) : 0.0f)) + beside;
            if (s != 5 && us < best.us) { best = TilePlan{i, s, us}; best_too = too; }
            if ((s != 5 || tiles * 6.0f > 256.0f) && too < other.us) other = TilePlan{i, s, too};
        }
    }
    if (rounds && ((other.form == best.form && other.splits < best.splits) || other.us * 1.1f <= best_too)) { best.form = other.form; best.splits = other.splits; }
    return best;
}
static void tell_plan(const DirectForm& f, const TilePlan& p, int* plan) { plan[0] = f.TM; plan[1] = f.TN; plan[2] = f.resident; plan[3] = p.splits; }

// the pieces of several matrices' columns side by side, in order, into each one's own results
template <int V>
__global__ __launch_bounds__(256) void gemm_direct_sum_kernel(const DirectArgs d) {
    const TileArgs& a = d.t;
    const int n = (blockIdx.x * 256 + threadIdx.x) * V, r = blockIdx.y;
    if (n >= a.N) return;
    const int n1 = d.seg_out[0], n2 = n1 + d.seg_out[1], sg = (n >= n1 ? 1 : 0) + (d.n_seg > 2 && n >= n2 ? 1 : 0);
    float* y = seg_pick(d.segY, sg) + (long long)r * seg_pick(d.seg_out, sg) + n - (sg == 0 ? 0 : sg == 1 ? n1 : n2);
    const float* p = a.part + (long long)r * a.N + n;
    float s[V] = {};
    for (int i = 0; i < a.splits; i += 4) {                 // four requests under way
        float v[4][V];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float* q = p + (long long)a.T * a.N * min(i + u, a.splits - 1);
            if constexpr (V == 4) { const float4 t = *reinterpret_cast<const float4*>(q); v[u][0] = t.x; v[u][1] = t.y; v[u][2] = t.z; v[u][3] = t.w; }
            else v[u][0] = *q;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u < a.splits)
#pragma unroll
                for (int j = 0; j < V; ++j) s[j] += v[u][j];
    }
    if constexpr (V == 4) *reinterpret_cast<float4*>(y) = float4{s[0], s[1], s[2], s[3]};
    else y[0] = s[0];
}

template <class P, int TM, int TN, int WM, int WN, int STAGES, int GLU, int MINW>
static int launch_direct(DirectArgs d, int splits, hipStream_t s, bool sum = true) {      // (as launch_tiles; without the sum several matrices' pieces lie as those of one of all their rows)
    constexpr int BK = 128 / (int)sizeof(typename P::WT);
    const int chunks = d.t.K / BK, per = (chunks + splits - 1) / splits;
    d.t.k_per_split = per * BK;
    d.t.splits = (chunks + per - 1) / per;
    const int row_tiles = d.t.offsets ? d.t.T / TM + d.t.G : (d.t.T + TM - 1) / TM;
    d.tile_rows = ((d.t.T + 15) / 16 + row_tiles - 1) / row_tiles * 16;
    int col_tiles = GLU ? (d.glu_ff + TN / 2 - 1) / (TN / 2) : (d.t.N + TN - 1) / TN;
    if (d.n_seg > 1) {
        col_tiles = 0;
        for (int i = 0; i < d.n_seg; ++i) { d.seg_tile[i] = col_tiles; col_tiles += (d.seg_out[i] + TN - 1) / TN; }
    }
    hipLaunchKernelGGL((gemm_direct_kernel<P, TM, TN, WM, WN, STAGES, GLU, MINW>), dim3(row_tiles * col_tiles * d.t.splits), dim3(64 * WM * WN), 0, s, d, row_tiles, col_tiles);
    if (d.t.splits == 1 || !sum) return d.t.splits;
    if (d.n_seg <= 1) { launch_tile_sum(d.t, s); return d.t.splits; }
    bool four = !((uintptr_t)d.t.part & 15);
    for (int i = 0; i < d.n_seg; ++i) four = four && d.seg_out[i] % 4 == 0 && !((uintptr_t)d.segY[i] & 15);
    if (four) hipLaunchKernelGGL((gemm_direct_sum_kernel<4>), dim3((d.t.N / 4 + 255) / 256, d.t.T), dim3(256), 0, s, d);
    else hipLaunchKernelGGL((gemm_direct_sum_kernel<1>), dim3((d.t.N + 255) / 256, d.t.T), dim3(256), 0, s, d);
    return d.t.splits;
}

}  // namespace ntk
