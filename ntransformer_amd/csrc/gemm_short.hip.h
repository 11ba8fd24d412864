// gemm_short.hip.h -- the launch of gemm_short.hip, for gemm_f16.hip's short prompts
#pragma once
#include "gemm_planes.hip.h"

namespace ntk {

constexpr int SS_TOKENS = 16;
struct ShortStreamSeg { const uint8_t* W; float* Y; float* part; int out, tile0; uint32_t p2_off; };      // as GemmBSeg
struct ShortStreamParams {
    ShortStreamSeg seg[3];
    int nseg;
    const uint8_t *xb, *aux;              // planes and step sums of the workspace's chunk
    const float *group_inv, *ssq;         // 1 / s of the groups of columns; rows' sums of squares in parts (X is divided by their roots), or null
    int nssq;
    float eps;
    const float* resid;                   // (one slice only)
    int T, in, units, ups, groups, tiles; // columns in units of 256: ups of them a slice (blockIdx.y), groups of row tiles a workgroup
};
struct ShortStreamPlan { int n = 0, ups = 0, groups = 0, wgx = 0; float us = 0.0f; };       // us: the estimate (n == 0: that of the other form)
// the slices of K (at most `most`); n == 0: the form with its planes in LDS is estimated to be ahead
ShortStreamPlan short_stream_plan(int dt, int units, int tiles, int most, int other);
// matrices of two formats (da < db as numbers: Q4_K, Q6_K, Q5_K) in one launch of equal slices; false: estimated behind two launches, which take `apart` us
bool short_stream_plan_two(int da, int db, int units, int tiles_a, int tiles_b, int most, float apart, ShortStreamPlan* a, ShortStreamPlan* b);
int short_stream_launch_two(int da, int db, const ShortStreamParams& a, const ShortStreamParams& b, const ShortStreamPlan& pa, const ShortStreamPlan& pb, hipStream_t st);
int short_stream_launch(int dt, const ShortStreamParams& p, const ShortStreamPlan& plan, hipStream_t st);

}  // namespace ntk
