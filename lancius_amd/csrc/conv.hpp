// What the convolution translation units share.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace lancius {

// The split-product convolution (conv_split.hip): out [N][C_out][Ho][Wo] from
// in [N][C_in][H][W] and the filter matrix wt.  Forward: out of a KH x KW
// convolution of `stride` and `pad`, wt [C_out][KH KW][C16].  dgrad: in = dy,
// out = dx of such a convolution (the names follow this product: C_in is dy's
// channels).  conv_split_fits says
// whether the sizes stay within the kernel's 32-bit offsets.
struct ConvSplitParams {
    float* out;
    const float* in;
    const float* wt;
    const float* bias;  // may be null
    int N, C_in, C16, H, W, C_out, KH, KW, stride, pad, Ho, Wo;  // C16: C_in rounded up to 16
    int dgrad, act;
    uint32_t tiles_m;  // set by the launch
    int small_tile;    // 16 or 32: conv2d_small's tile, 0: split products
};
// Time in us of the small-tile kernel with the better of its tiles.
double conv_small_plan(const ConvSplitParams& p, int* tile);
bool conv_split_fits(const ConvSplitParams& p);
size_t conv_split_weight_bytes(const ConvSplitParams& p);
size_t conv_split_tiles(const ConvSplitParams& p);  // workgroups of the launch
// w: the filter [out][in][KH][KW] to lay out first (null: p.wt is ready).
int launch_conv_split(lancius_hip_ctx* ctx, ConvSplitParams& p, const float* w);

// The split-product weight gradient (wgrad_split.hip): ws gets `splits` partial
// gradients [C_out][C_in KH KW], or dw the whole one when splits is 1.
struct WgradSplitParams {
    float* out;
    const float* dy;
    const float* x;
    int N, C_in, H, W, C_out, Ho, Wo, KH, KW, stride, pad;
    int J;          // C_in KH KW
    int row_oct;    // octets of 8 output pixels in a row, the last one padded
    int octets;     // N Ho row_oct
    int chunk;      // k-steps (two octets) per split
    int splits;
    uint32_t tiles_m, tiles_n;
};
// Sizes within its 32-bit offsets.
bool wgrad_split_fits(const WgradSplitParams& p);
// Sets chunk and splits for a grid of about one workgroup per CU; us: an estimate of the launch.
void wgrad_split_plan(WgradSplitParams& p, size_t cus, double* us);
bool wgrad_split_few(const WgradSplitParams& p);  // one range of few pixels
int launch_wgrad_split(lancius_hip_ctx* ctx, WgradSplitParams& p);

}  // namespace lancius
