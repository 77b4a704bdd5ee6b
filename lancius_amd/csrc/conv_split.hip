// Convolution and its input gradient on the bf16 matrix cores: an implicit
// GEMM (conv.hip) of split products (split.hpp, split_tile.hpp).
//
// GEMM view: Out[channel][P] = sum_k W[channel][k] X[k][P], k = (tap, channel
// of the input) with the channels padded to 16 in W (zeros), so a k-step of 16
// is one tap's run of channels.  W is a plain row-major matrix (RowLoader); a
// B-staging thread owns one pixel and loads its 16 channels a step, lanes
// along pixels: one offset a tap, the channels in the scalar offset.
//
// Input gradient: dx[ih] = sum_kh dy[(ih + pad - kh) / s] w[kh] over the kh
// that divide.  The pixels with (ih + pad) % s == a see the taps kh = a + s u
// only, at ho = (ih + pad - a) / s - u: each of the s x s classes is a
// convolution of stride 1 over its own taps, with no product spent on taps
// that miss (at stride 2 a quarter of the products of one convolution over
// the spread-out dy).
//
// Measured, fp32 kernels -> this: N32 64->128 3x3 56^2 131 -> 100 us forward,
// 142 -> 129 its gradient; N32 128->128 28^2 86 -> 49; the gradient at stride 2
// of N16 64->128 56^2 3263 (one thread an element) -> 32.  What bounds the
// first: 784 tiles on 512 slots, a second round half full; sharing the last
// tiles by k-steps through the point of coherence cost more than it saved (99
// -> 114 us: 512 shares of 64 KB of sums).  64 x 128 tiles read 9 KB of operands
// from LDS for 12 products a wave, 128 x 128 tiles 12 KB for 24.
#include <algorithm>
#include <cmath>

#include "conv.hpp"
#include "split_tile.hpp"

namespace lancius {
namespace {

__device__ __host__ __forceinline__ int taps_in_class(int k, int a, int s) { return a < k ? (k - a + s - 1) / s : 0; }

// One class's geometry: output pixel (th, tw) of th_n x tw_n lands at
// (os th + oh0, os tw + ow0) and reads the input at (mul th + h0 + dir uh,
// mul tw + w0 + dir uw) for taps uh < kh, uw < kw.
struct ConvClass {
    int th_n, tw_n, os, oh0, ow0, mul, h0, w0, dir, kh, kw;
    size_t w_off;  // floats before the class's filter matrix
};

__device__ __forceinline__ ConvClass conv_class(const ConvSplitParams& p, int z) {
    ConvClass c;
    if (!p.dgrad) {
        c = {p.Ho, p.Wo, 1, 0, 0, p.stride, -p.pad, -p.pad, 1, p.KH, p.KW, 0};
        return c;
    }
    const int s = p.stride, a = z / s, b = z - a * s;
    const int first_h = ((a - p.pad) % s + s) % s, first_w = ((b - p.pad) % s + s) % s;
    c.th_n = first_h < p.Ho ? (p.Ho - first_h + s - 1) / s : 0;
    c.tw_n = first_w < p.Wo ? (p.Wo - first_w + s - 1) / s : 0;
    c.os = s;
    c.oh0 = first_h;
    c.ow0 = first_w;
    c.mul = 1;
    c.h0 = (first_h + p.pad - a) / s;
    c.w0 = (first_w + p.pad - b) / s;
    c.dir = -1;
    c.kh = taps_in_class(p.KH, a, s);
    c.kw = taps_in_class(p.KW, b, s);
    int before = 0;  // taps of the classes before this one
    for (int i = 0; i < z; ++i) before += taps_in_class(p.KH, i / s, s) * taps_in_class(p.KW, i % s, s);
    c.w_off = (size_t)before * p.C16 * p.C_out;
    return c;
}

// B's loader: a pixel's 16 channels of a step, chunk c its channels 8 c ..
template <int BN, int KG>
struct PixelLoader {
    __amdgpu_buffer_rsrc_t rs;
    int wr[2], hb, wb, dir, H, W, C16, kw, hw4, img, c0, uh, uw, kh;
    f32x8 s[2];
    bool valid;
    __device__ __forceinline__ void skip(int channels) {
        c0 += channels;
        while (c0 >= C16) {
            c0 -= C16;
            if (++uw == kw) {
                uw = 0;
                ++uh;
            }
        }
    }
    __device__ __forceinline__ void load() {
        const int hi = hb + dir * uh, wi = wb + dir * uw;
        const bool in = valid & (uh < kh) & ((unsigned)hi < (unsigned)H) & ((unsigned)wi < (unsigned)W);
        const int off = pick(in, img + (hi * W + wi) * 4, 0x7ffffff0);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                s[c][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, (c0 + 8 * c + i) * hw4, 0));
        skip(16 * KG);
    }
    __device__ __forceinline__ f32x8 chunk(int c) const { return s[c]; }
};

template <int BM, int BN, int WM, int WN, int KG>
__global__ void __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG, 2) conv2d_split(const ConvSplitParams p) {
    using T = SplitTile<BM, BN, WM, WN, KG, kTwoSums, 3>;
    constexpr int TN = T::TN;
    static_assert(T::CB == 2, "a thread stages both k halves of a pixel");
    __shared__ __attribute__((aligned(16))) char smem[T::SMEM];
    const ConvClass cl = conv_class(p, blockIdx.z);
    const int pix_img = cl.th_n * cl.tw_n, P_n = p.N * pix_img;
    const uint32_t tiles_n = (uint32_t)((P_n + BN - 1) / BN);
    if (blockIdx.x >= p.tiles_m * tiles_n) return;  // a class of fewer pixels than the largest
    uint32_t tm_id, tn_id;
    grouped_tile(xcd_contiguous_id(blockIdx.x, p.tiles_m * tiles_n), p.tiles_m, tiles_n, 2, tm_id, tn_id);
    const int m0 = (int)tm_id * BM, P0 = (int)tn_id * BN;
    const int K = cl.kh * cl.kw * p.C16;
    const int hw4 = p.H * p.W * 4;
    const float* __restrict__ wt = p.wt + cl.w_off;
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(wt), 0, p.C_out * K * 4, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.in), 0, p.N * p.C_in * hw4, kBufferRsrcWord3);
    constexpr int kOut = 0x7ffffff0;

    T t;
    t.clear();
    const int iters = (K / 16 + KG - 1) / KG;
    if (K == 0) {
        // a class that no tap reaches: its pixels are 0
    } else if (t.stages_a()) {
        RowLoader<BM, T::CA, KG, false> ld(rw, t.stager(), m0, K, t.grp * 16);
        t.template run<true>(smem, ld, iters);
    } else {
        PixelLoader<BN, KG> ld{rx};
        const int st = t.stager(), P = P0 + st;
        ld.valid = P < P_n;
        const int n = P / pix_img, rem = P - n * pix_img, th = rem / cl.tw_n, tw = rem - th * cl.tw_n;
        ld.wr[0] = st * 16;
        ld.wr[1] = (BN + st) * 16;
        ld.hb = cl.mul * th + cl.h0;
        ld.wb = cl.mul * tw + cl.w0;
        ld.dir = cl.dir;
        ld.H = p.H;
        ld.W = p.W;
        ld.C16 = p.C16;
        ld.kh = cl.kh;
        ld.kw = cl.kw;
        ld.hw4 = hw4;
        ld.img = n * p.C_in * hw4;
        ld.c0 = ld.uh = ld.uw = 0;
        ld.skip(16 * t.grp);
        t.template run<false>(smem, ld, iters);
    }
    t.reduce(smem);

    // this lane's pixels of each block column: byte offsets in the output
    const int ohw4 = p.Ho * p.Wo * 4;
    int po[TN], px[TN], py[TN], pn[TN];
    bool ok[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int P = P0 + t.wn * WN + 32 * j + t.lr;
        ok[j] = P < P_n;
        const int n = P / pix_img, rem = P - n * pix_img;
        pn[j] = n;
        py[j] = rem / cl.tw_n;
        px[j] = rem - py[j] * cl.tw_n;
        po[j] = n * p.C_out * ohw4 + ((cl.os * py[j] + cl.oh0) * p.Wo + cl.os * px[j] + cl.ow0) * 4;
    }
    const int mw = m0 + t.row0();

    // sums that are not all finite are recomputed in fp32 (split.hpp)
    if (t.not_finite())
        t.recompute(
            0, K,
            [&](int i, int k) {
                const int row = mw + 32 * i + t.lr;
                return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                     rw, pick((row < p.C_out) & (k < K), (row * K + k) * 4, kOut), 0, 0));
            },
            [&](int j, int k) {  // (four channels of one tap: C16 is a multiple of 16)
                const int tap = k / p.C16, c = k - tap * p.C16, uh = tap / cl.kw, uw = tap - uh * cl.kw;
                const int hi = cl.mul * py[j] + cl.h0 + cl.dir * uh, wi = cl.mul * px[j] + cl.w0 + cl.dir * uw;
                const bool in = ok[j] & (k < K) & ((unsigned)hi < (unsigned)p.H) & ((unsigned)wi < (unsigned)p.W);
                const int off = (pn[j] * p.C_in + c) * hw4 + (hi * p.W + wi) * 4;
                f32x4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                         rx, pick(in & (c + q < p.C_in), off + q * hw4, kOut), 0, 0));
                return v;
            });

    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, p.N * p.C_out * ohw4, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.bias), 0, p.bias ? p.C_out * 4 : 0, kBufferRsrcWord3);
    const bool relu = p.act == kActRelu;
#pragma unroll
    for (int i = 0; i < T::TS; ++i) {
        const int c0 = mw + 32 * i + 4 * t.lk;  // channel of register r: c0 + 8 (r / 4) + r % 4
        float bv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            bv[r] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(rb, c0 * 4, (8 * (r >> 2) + (r & 3)) * 4, 0));
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int q = 8 * (r >> 2) + (r & 3);
                const float v = t.acc[i][j][r] + bv[r], w = relu ? relu_ref(v) : v;
                const int o = pick(ok[j] & (c0 + q < p.C_out), po[j] + c0 * ohw4, kOut);
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w), ro, o, q * ohw4, 0);
            }
    }
}

// The same product in fp32 for grids that leave most CUs idle: a tile of T
// channels x T pixels per workgroup, K spread over its waves, operands loaded
// straight into the matrix cores' registers (gemm_small.hip's scheme). What
// bounds it is a wave's chain of gathers, what bounded the staged tiles the
// same chain for 128 pixels with a barrier a step. Before and now: N32 16->32
// 5x5 16^2 15.8, 5.5 us, its input gradient 28, 10.4; N1 64->128 3x3 56^2 23.5,
// 9.6; N3 176->16 5x5 of 8x9 115, 14.
template <int T, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) conv2d_small(const ConvSplitParams p) {
    constexpr int NQ = T * T / 64;                // sums a lane holds
    constexpr int KS = 4 * (64 / T);              // k of a group: four MFMAs
    constexpr int NACC = T == 32 ? 2 : 4;
    constexpr int kOut = 0x7ffffff0;
    __shared__ float red[WAVES][NQ][64];
    const ConvClass cl = conv_class(p, blockIdx.z);
    const int pix_img = cl.th_n * cl.tw_n, P_n = p.N * pix_img;
    const uint32_t tiles_n = (uint32_t)((P_n + T - 1) / T);
    if (blockIdx.x >= p.tiles_m * tiles_n) return;  // a class of fewer pixels than the largest
    const int m0 = (int)(blockIdx.x % p.tiles_m) * T, P0 = (int)(blockIdx.x / p.tiles_m) * T;
    const int K = cl.kh * cl.kw * p.C16;
    const int hw4 = p.H * p.W * 4;
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.wt + cl.w_off), 0, p.C_out * K * 4, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.in), 0, p.N * p.C_in * hw4, kBufferRsrcWord3);
    const int lane = threadIdx.x & 63, lr = lane % T, lk = lane / T;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    // this lane's pixel
    const int P = P0 + lr;
    const bool valid = P < P_n;
    const int n = P / pix_img, rem = P - n * pix_img, th = rem / cl.tw_n, tw = rem - th * cl.tw_n;
    const int hb = cl.mul * th + cl.h0, wb = cl.mul * tw + cl.w0;
    const int img = n * p.C_in * hw4;

    // this wave's groups [gi, ge), the next one to load at (tap uh uw, channels c0..)
    const int groups = K / KS, per = (groups + WAVES - 1) / WAVES;
    int gi = wave * per;
    const int ge = min(groups, gi + per);
    int tap = gi * KS / p.C16, c0 = gi * KS - tap * p.C16, k0 = gi * KS;
    int uh = cl.kw ? tap / cl.kw : 0, uw = tap - uh * cl.kw;
    typedef float acc_t __attribute__((ext_vector_type(NQ)));
    f32x4 a[2], b[2];
    acc_t acc[NACC] = {};  // by k modulo NACC: short chains, and no MFMA waits for the one before
    auto load = [&](int s) {
        const int hi = hb + cl.dir * uh, wi = wb + cl.dir * uw, c = c0 + 4 * lk;
        const bool in = valid & ((unsigned)hi < (unsigned)p.H) & ((unsigned)wi < (unsigned)p.W);
        const int off = img + (hi * p.W + wi) * 4 + 4 * lk * hw4;
#pragma unroll
        for (int j = 0; j < 4; ++j)  // (channels past C_in are the next image's)
            b[s][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                    rx, pick(in & (c + j < p.C_in), off, kOut), (c0 + j) * hw4, 0));
        a[s] = __builtin_bit_cast(f32x4,
                                  __builtin_amdgcn_raw_buffer_load_b128(rw, ((m0 + lr) * K + 4 * lk) * 4, k0 * 4, 0));
        k0 += KS;
        c0 += KS;
        if (c0 == p.C16) {
            c0 = 0;
            if (++uw == cl.kw) {
                uw = 0;
                ++uh;
            }
        }
    };
    auto multiply = [&](int s) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            acc_t& c = acc[j % NACC];
            if constexpr (T == 32)
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s][j], b[s][j], c, 0, 0, 0);
            else
                c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][j], b[s][j], c, 0, 0, 0);
        }
    };
    if (gi < ge) {
        load(0);
        for (; gi + 2 < ge; gi += 2) {
            load(1);
            multiply(0);
            load(0);
            multiply(1);
        }
        if (gi + 1 < ge) {
            load(1);
            multiply(0);
            multiply(1);
        } else {
            multiply(0);
        }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        float s = acc[0][q] + acc[1][q];
        if constexpr (NACC == 4) s += acc[2][q] + acc[3][q];
        red[wave][q][lane] = s;
    }
    __syncthreads();

    // element (q, lane): pixel lane % T, channel 8 (q / 4) + 4 (lane / T) + q % 4
    const int ohw = p.Ho * p.Wo;
    float* __restrict__ out = p.out + (size_t)n * p.C_out * ohw + (cl.os * th + cl.oh0) * p.Wo + cl.os * tw + cl.ow0;
    const bool relu = p.act == kActRelu;
#pragma unroll
    for (int q0 = 0; q0 < NQ; q0 += WAVES) {
        const int q = q0 + wave, c = m0 + 8 * (q >> 2) + 4 * lk + (q & 3);
        if (q < NQ && valid && c < p.C_out) {
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) s += red[w][q][lane];
            if (p.bias) s += p.bias[c];
            out[(size_t)c * ohw] = relu ? relu_ref(s) : s;
        }
    }
}

// wt[channel][tap][C16]: the forward filter re-laid, channels past C_in zero.
__global__ void __launch_bounds__(256) conv_split_weights(float* __restrict__ wt, const float* __restrict__ w, int C_out,
                                                          int C_in, int C16, int KHW) {
    const size_t total = (size_t)C_out * KHW * C16;
    for (size_t d = (size_t)blockIdx.x * 256 + threadIdx.x; d < total; d += (size_t)gridDim.x * 256) {
        const int ci = (int)(d % C16);
        const size_t r = d / C16;
        const int tap = (int)(r % KHW), co = (int)(r / KHW);
        wt[d] = ci < C_in ? w[((size_t)co * C_in + ci) * KHW + tap] : 0.0f;
    }
}

// The input gradient's filter matrices, one per class: [ci][tap of the class][co
// padded to C16].  w is the forward filter [F_out][F_in][KH][KW].
__global__ void __launch_bounds__(256) dgrad_split_weights(float* __restrict__ wt, const float* __restrict__ w, int F_out,
                                                           int F_in, int C16, int KH, int KW, int s) {
    const size_t total = (size_t)F_in * KH * KW * C16;
    for (size_t d = (size_t)blockIdx.x * 256 + threadIdx.x; d < total; d += (size_t)gridDim.x * 256) {
        size_t left = d;
        int z = 0, kh_n = 0, kw_n = 0;
        for (;; ++z) {
            kh_n = taps_in_class(KH, z / s, s);
            kw_n = taps_in_class(KW, z % s, s);
            const size_t n = (size_t)F_in * kh_n * kw_n * C16;
            if (left < n) break;
            left -= n;
        }
        const int co = (int)(left % C16);
        const size_t r = left / C16;
        const int tap = (int)(r % (kh_n * kw_n)), ci = (int)(r / (kh_n * kw_n));
        const int kh = z / s + s * (tap / kw_n), kw = z % s + s * (tap % kw_n);
        wt[d] = co < F_out ? w[(((size_t)co * F_in + ci) * KH + kh) * KW + kw] : 0.0f;
    }
}

template <int BM, int BN, int WM, int WN, int KG>
int launch(lancius_hip_ctx* ctx, ConvSplitParams& p, size_t P_max, unsigned classes) {
    p.tiles_m = (uint32_t)((p.C_out + BM - 1) / BM);
    const size_t tiles = p.tiles_m * ((P_max + BN - 1) / BN);
    hipLaunchKernelGGL((conv2d_split<BM, BN, WM, WN, KG>), dim3((unsigned)tiles, 1, classes),
                       dim3(64 * (BM / WM) * (BN / WN) * KG), 0, ctx->stream, p);
    return check_launch(LANCIUS_KERNEL_NAME("conv2d_split %dx%d x%d", BM, BN, KG));
}

template <int T, int WAVES>
int launch_small(lancius_hip_ctx* ctx, ConvSplitParams& p, size_t P_max, unsigned classes) {
    p.tiles_m = (uint32_t)((p.C_out + T - 1) / T);
    const size_t tiles = p.tiles_m * ((P_max + T - 1) / T);
    hipLaunchKernelGGL((conv2d_small<T, WAVES>), dim3((unsigned)tiles, 1, classes), dim3(64 * WAVES), 0, ctx->stream, p);
    return check_launch(LANCIUS_KERNEL_NAME("conv2d_small %dx%d", T, T));
}

}  // namespace

bool conv_split_fits(const ConvSplitParams& p) {
    constexpr size_t lim = (size_t)1 << 31;
    const size_t in = (size_t)p.H * p.W * 4, out = (size_t)p.Ho * p.Wo * 4;
    // (an offset past the end of any of them, 0x7ffffff0, takes at most 27
    // output planes or the input's channels more before it would wrap)
    return (size_t)p.N * p.C_in * in < lim - 64 && (size_t)p.C16 * in < lim - 64 && (size_t)p.N * p.C_out * out < lim - 64 &&
           out < ((size_t)1 << 26) && (size_t)p.N * p.Ho * p.Wo < lim - 256 &&
           (size_t)(p.C_out + 128) * p.KH * p.KW * p.C16 * 4 < lim - 64;
}

size_t conv_split_weight_bytes(const ConvSplitParams& p) {
    return (size_t)p.C_out * p.KH * p.KW * p.C16 * sizeof(float);
}

namespace {

int launch_conv_split_weights(lancius_hip_ctx* ctx, const ConvSplitParams& p, float* wt, const float* w) {
    const size_t total = conv_split_weight_bytes(p) / sizeof(float);
    const dim3 grid((unsigned)std::min<size_t>((total + 255) / 256, 2048));
    if (p.dgrad)
        hipLaunchKernelGGL(dgrad_split_weights, grid, dim3(256), 0, ctx->stream, wt, w, p.C_in, p.C_out, p.C16, p.KH,
                           p.KW, p.stride);
    else
        hipLaunchKernelGGL(conv_split_weights, grid, dim3(256), 0, ctx->stream, wt, w, p.C_out, p.C_in, p.C16,
                           p.KH * p.KW);
    return check_launch("conv_split_weights");
}

}  // namespace

size_t conv_split_tiles(const ConvSplitParams& p) {
    const size_t s = p.dgrad ? (size_t)p.stride : 1;
    const size_t pixels = (size_t)p.N * ((p.Ho + s - 1) / s) * ((p.Wo + s - 1) / s);
    return s * s * (p.C_out <= 64 ? 1 : (p.C_out + 127) / 128) * ((pixels + 127) / 128);
}

// Fitted to 220 convolutions and gradients of up to 110 images' rows a side
// (15 % rms): a wave's chain of K, a cost a tile, the operands a tile reads.
// Beyond 20 us the fit is short of ragged and strided gathers.
double conv_small_plan(const ConvSplitParams& p, int* tile) {
    const size_t s = p.dgrad ? (size_t)p.stride : 1;
    const double pixels = (double)p.N * (double)((p.Ho + s - 1) / s) * (double)((p.Wo + s - 1) / s);
    const double taps = (double)((p.KH + s - 1) / s) * (double)((p.KW + s - 1) / s);
    const double k_max = taps * p.C16, k = (double)p.KH * p.KW * p.C16 / (double)(s * s);
    auto tiles = [&](double t) { return (double)(s * s) * std::ceil(p.C_out / t) * std::ceil(pixels / t); };
    const double us16 = 1.5 + 2.9e-3 * k_max + tiles(16) * (3.1e-3 + 1.05e-5 * k);
    const double us32 = 2.3 + 5.3e-3 * k_max + tiles(32) * (5.2e-3 + 2.05e-5 * k);
    *tile = us16 <= us32 ? 16 : 32;
    const double us = std::max(4.7, std::min(us16, us32));
    return us + 0.7 * std::max(0.0, us - 20.0);
}

int launch_conv_split(lancius_hip_ctx* ctx, ConvSplitParams& p, const float* w) {
    if (w) {
        void* ws = nullptr;
        if (int rc = workspace(ctx, conv_split_weight_bytes(p), &ws)) return rc;
        if (int rc = launch_conv_split_weights(ctx, p, (float*)ws, w)) return rc;
        p.wt = (const float*)ws;
    }
    const size_t s = p.dgrad ? (size_t)p.stride : 1;
    const size_t pixels = (size_t)p.N * ((p.Ho + s - 1) / s) * ((p.Wo + s - 1) / s);
    const unsigned classes = (unsigned)(s * s);
    if (p.small_tile == 32) return launch_small<32, 8>(ctx, p, pixels, classes);
    if (p.small_tile == 16) return launch_small<16, 8>(ctx, p, pixels, classes);
    // 128 channels x 128 pixels, or 64 x 128 for at most 64 channels: four
    // waves, two workgroups a CU; grids of at most one tile a CU give each
    // tile eight waves in two k-groups
    const bool kg2 = conv_split_tiles(p) <= (size_t)cu_count(ctx);
    if (p.C_out <= 64)
        return kg2 ? launch<64, 128, 64, 32, 2>(ctx, p, pixels, classes) : launch<64, 128, 64, 32, 1>(ctx, p, pixels, classes);
    return kg2 ? launch<128, 128, 64, 64, 2>(ctx, p, pixels, classes) : launch<128, 128, 64, 64, 1>(ctx, p, pixels, classes);
}

}  // namespace lancius
