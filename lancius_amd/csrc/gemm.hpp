// What the GEMM translation units share.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace lancius {

struct GemmParams {
    float* C[LANCIUS_HIP_MAX_GROUP];
    const float* A[LANCIUS_HIP_MAX_GROUP];
    const float* R[LANCIUS_HIP_MAX_GROUP];     // residuals (may be null)
    const float* B[LANCIUS_HIP_MAX_GROUP];
    const float* bias[LANCIUS_HIP_MAX_GROUP];  // may be null
    int M, N, K;
    int act;
    uint32_t tiles_m, tiles_n;
    float* ws;   // split-K partials [count][splits][M][N]
    unsigned* counters;  // fused skinny split-K: one arrival counter per (group, column block), zero between launches
    int splits;  // K ranges (blockIdx.y), 1 = no split
    int kchunk;  // K per split, a multiple of the k-tile
};

// Tiles of the split-product kernels (gemm_split.hip), by cost per launch.
enum : int { kSplit256, kSplit256x128, kSplit128 };
// Launches one: p.splits and p.kchunk (a multiple of 32) set, splits > 1 with
// kSplit128 only, partial sums to p.ws for the caller to add; not both
// operands transposed, operands and C each under kSplitMaxBytes.
int launch_gemm_split(lancius_hip_ctx* ctx, GemmParams& p, int count, bool ta, bool tb, int tile);
// Buffer offsets are 32-bit; they run up to 96 k past an operand's end and
// 256 rows past C's.
constexpr size_t kSplitMaxBytes = (size_t)1 << 31;

// gemm_small.hip: the tile (16 or 32) and cost of a product in one launch of
// small tiles, and that launch; operands and C within split_fits' bounds.
struct SmallPlan {
    int tile;
    double us;
};
SmallPlan gemm_small_plan(size_t count, size_t M, size_t K, size_t N, bool tb);
int launch_gemm_small(lancius_hip_ctx* ctx, GemmParams& p, int count, bool ta, bool tb, int tile);

}  // namespace lancius
