// Weight gradient of a convolution on the bf16 matrix cores (split.hpp,
// split_tile.hpp):
//   dW[co][j] = sum_P dY[co][P] X[j][P],  j = (ci, kh, kw), P = (n, ho, wo).
//
// Both operands run along the pixels, so a chunk of 8 k is 8 output pixels of
// one row (an octet; the last of a row padded, dY cleared past its end): 32
// contiguous bytes of dY, and at stride 1 of X too, shifted by the tap.  X is
// cleared outside the image; which row and column an octet has is kept as
// (image, row, octet) and advanced without a division.  K is split over
// workgroups, one of eight waves in two k-groups per CU, whose partial
// gradients wgrad_reduce (conv.hip) adds in order.
//
// N32 64->128 3x3 56^2 (5 tiles of 128 x 128, 51 ranges of 123 steps): fp32
// kernel 143 us, this 98 (matrix cores busy 0.51 of the busy CUs' cycles, the
// vector unit 0.54: X's addresses, masks and splits); N32 256->256 14^2 87 -> 58.
#include <algorithm>

#include "conv.hpp"
#include "split_tile.hpp"

namespace lancius {
namespace {

constexpr int kOut = 0x7ffffff0;  // past the end of any operand: the load returns 0

// Octet o of the reduction as (image, row, octet of the row), stepped by 2 KG.
struct Octet {
    int n, ho, w8, o, end;
    int dn, dh, dw, row_oct, Ho, by;
    __device__ __forceinline__ Octet(const WgradSplitParams& p, int first, int last, int step) {
        row_oct = p.row_oct;
        Ho = p.Ho;
        o = first;
        end = last;
        by = step;
        w8 = first % row_oct;
        const int r = first / row_oct;
        ho = r % Ho;
        n = r / Ho;
        dw = step % row_oct;
        dh = step / row_oct % Ho;
        dn = step / row_oct / Ho;
    }
    __device__ __forceinline__ void next() {
        o += by;
        w8 += dw;
        ho += dh;
        n += dn;
        if (w8 >= row_oct) {
            w8 -= row_oct;
            ++ho;
        }
        if (ho >= Ho) {
            ho -= Ho;
            ++n;
        }
    }
};

// dY rows krow (and krow + BE/2): 8 pixels.
template <int BE, int CN>
struct DyLoader {
    __amdgpu_buffer_rsrc_t rs;
    Octet q;
    int wr[CN], row[CN], Wo, img, left;
    f32x8 s[CN];
    __device__ __forceinline__ DyLoader(__amdgpu_buffer_rsrc_t rs_, const WgradSplitParams& p, int st, int m0, Octet q_)
        : rs(rs_), q(q_) {
        const int kh = (st >> 5) & 1, r = (st & 31) + 32 * (st >> 6);
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            wr[c] = (kh * BE + r + c * (BE / 2)) * 16;
            row[c] = (m0 + r + c * (BE / 2)) * p.Ho * p.Wo * 4;
        }
        Wo = p.Wo;
        img = p.C_out * p.Ho * p.Wo * 4;
    }
    __device__ __forceinline__ void load() {
        const int base = q.n * img + (q.ho * Wo + 8 * q.w8) * 4;
        left = q.o < q.end ? Wo - 8 * q.w8 : 0;
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            const int off = pick(q.o < q.end, base + row[c], kOut);
            const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
            const f32x4 y = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 16, 0));
            s[c] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        q.next();
    }
    __device__ __forceinline__ f32x8 chunk(int c) const {
        f32x8 x = s[c];
        if (Wo & 7) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = i < left ? x[i] : 0.0f;
        }
        return x;
    }
};

// X rows j (and j + BE/2): the octet's 8 pixels seen through tap (kh, kw) of
// channel ci.  S1: stride 1, eight contiguous values.
template <int BE, int CN, bool S1>
struct XLoader {
    __amdgpu_buffer_rsrc_t rs;
    Octet q;
    int wr[CN], ch[CN], dh[CN], dwx[CN], wi[CN], H, W, stride, img;
    f32x8 s[CN];
    __device__ __forceinline__ XLoader(__amdgpu_buffer_rsrc_t rs_, const WgradSplitParams& p, int st, int j0, Octet q_)
        : rs(rs_), q(q_) {
        const int kh = (st >> 5) & 1, r = (st & 31) + 32 * (st >> 6), khw = p.KH * p.KW;
        H = p.H;
        W = p.W;
        stride = p.stride;
        img = p.C_in * H * W;
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            wr[c] = (kh * BE + r + c * (BE / 2)) * 16;
            const int j = min(j0 + r + c * (BE / 2), p.J - 1);  // (columns past J are never stored)
            const int ci = j / khw, t = j - ci * khw, th = t / p.KW;
            ch[c] = ci * H * W;
            dh[c] = th - p.pad;
            dwx[c] = t - th * p.KW - p.pad;
        }
    }
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            const int hi = q.ho * stride + dh[c];
            const bool in = (q.o < q.end) & ((unsigned)hi < (unsigned)H);
            const int base = q.n * img + ch[c] + hi * W;
            if constexpr (S1) {
                wi[c] = 8 * q.w8 + dwx[c];
                const int at = base + wi[c];
                const int off = pick(in & (at >= 0), at * 4, kOut);
                const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
                const f32x4 y = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 16, 0));
                s[c] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
                // an octet that starts left of the very first value of x
                if (__any(in & (at < 0))) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float v = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(rs, pick(at + i >= 0, (at + i) * 4, kOut), 0, 0));
                        s[c][i] = at < 0 ? v : s[c][i];
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int w = (8 * q.w8 + i) * stride + dwx[c];
                    const int off = pick(in & ((unsigned)w < (unsigned)W), (base + w) * 4, kOut);
                    s[c][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
                }
            }
        }
        q.next();
    }
    __device__ __forceinline__ f32x8 chunk(int c) const {
        f32x8 x = s[c];
        if constexpr (S1) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = (unsigned)(wi[c] + i) < (unsigned)W ? x[i] : 0.0f;
        }
        return x;
    }
};

template <int BM, int BN, int WM, int WN, int KG, bool S1>
__global__ void __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG, 2) wgrad_split(const WgradSplitParams p) {
    using T = SplitTile<BM, BN, WM, WN, KG, kTwoSums, 0>;
    constexpr int TN = T::TN;
    __shared__ __attribute__((aligned(16))) char smem[T::SMEM];
    const int m0 = (int)(blockIdx.x / p.tiles_n) * BM, j0 = (int)(blockIdx.x % p.tiles_n) * BN;
    const int HWo = p.Ho * p.Wo;
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.dy), 0, p.N * p.C_out * HWo * 4, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.x), 0, p.N * p.C_in * p.H * p.W * 4, kBufferRsrcWord3);
    const int o_begin = (int)blockIdx.y * p.chunk * 2, o_end = min(p.octets, o_begin + 2 * p.chunk);

    T t;
    t.clear();
    const int st = t.stager();
    const Octet q(p, o_begin + 2 * t.grp + ((st >> 5) & 1), o_end, 2 * KG);
    const int iters = ((o_end - o_begin + 1) / 2 + KG - 1) / KG;
    if (t.stages_a()) {
        DyLoader<BM, T::CA> ld(ra, p, st, m0, q);
        t.template run<true>(smem, ld, iters);
    } else {
        XLoader<BN, T::CB, S1> ld(rb, p, st, j0, q);
        t.template run<false>(smem, ld, iters);
    }
    t.reduce(smem);
    const int mw = m0 + t.row0();

    // sums that are not all finite are recomputed in fp32 (split.hpp)
    if (t.not_finite()) {
        struct Pixel {
            int n, ho, wo;
            bool in;
        };
        auto pixel = [&](int k) {  // the first of four in one octet
            const int o = k >> 3, r = o / p.row_oct, n = r / p.Ho;
            return Pixel{n, r - n * p.Ho, 8 * (o - r * p.row_oct) + (k & 7), o < o_end};
        };
        t.recompute(
            8 * o_begin, 8 * o_end,
            [&](int i, int k) {
                const Pixel x = pixel(k);
                const int co = mw + 32 * i + t.lr;
                const int off = ((x.n * p.C_out + co) * HWo + x.ho * p.Wo + x.wo) * 4;
                f32x4 v = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, pick(x.in & (co < p.C_out), off, kOut), 0, 0));
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = x.wo + q < p.Wo ? v[q] : 0.0f;
                return v;
            },
            [&](int j, int k) {
                const Pixel x = pixel(k);
                const int col = min(j0 + t.wn * WN + 32 * j + t.lr, p.J - 1), khw = p.KH * p.KW;
                const int ci = col / khw, tap = col - ci * khw, th = tap / p.KW, tw = tap - th * p.KW;
                const int hi = x.ho * p.stride + th - p.pad;
                const bool row = x.in & ((unsigned)hi < (unsigned)p.H);
                const int base = ((x.n * p.C_in + ci) * p.H + hi) * p.W;
                f32x4 v;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int wi = (x.wo + q) * p.stride + tw - p.pad;
                    const bool in = row & (x.wo + q < p.Wo) & ((unsigned)wi < (unsigned)p.W);
                    v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, pick(in, (base + wi) * 4, kOut), 0, 0));
                }
                return v;
            });
    }

    // rows past C_out fall past the end of this split's gradient
    float* const out = p.out + (size_t)blockIdx.y * p.C_out * p.J;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(out, 0, p.C_out * p.J * 4, kBufferRsrcWord3);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = j0 + t.wn * WN + 32 * j + t.lr;
        const int o = pick(col < p.J, ((mw + 4 * t.lk) * p.J + col) * 4, kOut);
#pragma unroll
        for (int i = 0; i < T::TS; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (float)t.acc[i][j][r]), ro, o,
                                                      (32 * i + 8 * (r >> 2) + (r & 3)) * p.J * 4, 0);
    }
}

template <int BM, int BN, int WM, int WN, int KG>
void launch(hipStream_t stream, const WgradSplitParams& p) {
    const dim3 grid(p.tiles_m * p.tiles_n, (unsigned)p.splits), block(64 * (BM / WM) * (BN / WN) * KG);
    if (p.stride == 1)
        hipLaunchKernelGGL((wgrad_split<BM, BN, WM, WN, KG, true>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((wgrad_split<BM, BN, WM, WN, KG, false>), grid, block, 0, stream, p);
}

}  // namespace

bool wgrad_split_fits(const WgradSplitParams& p) {
    constexpr size_t lim = (size_t)1 << 31;
    return (size_t)p.N * p.C_out * p.Ho * p.Wo * 4 < lim - 64 && (size_t)(p.C_out + 128) * p.Ho * p.Wo * 4 < lim - 64 &&
           (size_t)p.N * p.C_in * p.H * p.W * 4 < lim - 64 && (size_t)(p.C_out + 256) * p.J * 4 < lim - 64 &&
           (size_t)(p.J + 128) * 128 * 4 < lim && (size_t)p.N * p.Ho * ((p.Wo + 7) / 8) < ((size_t)1 << 27) &&
           p.stride < (1 << 15) && p.pad < (1 << 15) && (size_t)p.Wo * p.stride < ((size_t)1 << 30) &&
           (size_t)p.Ho * p.stride < ((size_t)1 << 30);
}

bool wgrad_split_few(const WgradSplitParams& p) { return p.splits == 1 && p.chunk <= 32; }

void wgrad_split_plan(WgradSplitParams& p, size_t cus, double* us) {
    p.row_oct = (p.Wo + 7) / 8;
    p.octets = p.N * p.Ho * p.row_oct;
    const size_t bm = p.C_out > 64 ? 128 : 64;
    p.tiles_m = (uint32_t)((p.C_out + bm - 1) / bm);
    p.tiles_n = (uint32_t)((p.J + 127) / 128);
    const size_t tiles = (size_t)p.tiles_m * p.tiles_n, steps = (size_t)(p.octets + 1) / 2;
    // ranges of K for one workgroup per CU, each at least 16 steps
    size_t splits = std::max<size_t>(1, std::min(cus / std::max<size_t>(tiles, 1), steps / 16));
    while (splits > 1 && splits * p.C_out * p.J * sizeof(float) > ((size_t)1 << 28)) splits = (splits + 1) / 2;
    p.chunk = (int)((steps + splits - 1) / splits);
    p.chunk += p.chunk & 1;  // both k-groups take as many steps
    p.splits = (int)((steps + p.chunk - 1) / p.chunk);
    const double rounds = (double)((tiles * p.splits + cus - 1) / cus);
    const double parts = p.splits > 1 ? 3.0 + 4.0 * p.C_out * p.J * p.splits * 2.0 / 4e6 : 0.0;
    *us = rounds * (8.0 + (bm == 128 ? 0.68 : 0.4) * p.chunk) + parts;
    // one short range: two steps 5.4 us (7.0), sixteen 12.4 (16.5), thirty 20
    if (wgrad_split_few(p) && rounds == 1.0) *us = bm == 128 ? 5.6 + 0.69 * p.chunk : 4.4 + 0.5 * p.chunk;
}

int launch_wgrad_split(lancius_hip_ctx* ctx, WgradSplitParams& p) {
    if (p.C_out > 64)
        launch<128, 128, 64, 64, 2>(ctx->stream, p);
    else
        launch<64, 128, 64, 32, 2>(ctx->stream, p);
    return check_launch(p.C_out > 64 ? "wgrad_split 128x128" : "wgrad_split 64x128");
}

}  // namespace lancius
