// fp32 GEMM on the bf16 matrix cores: both operands are split into three bf16
// parts on the way into LDS and multiplied as six bf16 products (split.hpp,
// split_tile.hpp).
#include "gemm.hpp"
#include "split_tile.hpp"

namespace lancius {
namespace {

// One BM x BN tile of C per workgroup.
template <int BM, int BN, int WM, int WN, int KG, bool TA, bool TB, bool SPLIT, int MODE, int SCHED>
__global__ void __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG, 2) gemm_f32_split(const GemmParams p) {
    using T = SplitTile<BM, BN, WM, WN, KG, MODE, SCHED>;
    constexpr int TN = T::TN, BK = T::BK;
    __shared__ __attribute__((aligned(16))) char smem[T::SMEM];

    const int g = blockIdx.z;
    const float* __restrict__ A = p.A[g];
    const float* __restrict__ B = p.B[g];
    float* __restrict__ C = p.C[g];
    const float* __restrict__ R = p.R[g];
    const int M = p.M, N = p.N, K = p.K;
    uint32_t tm_id, tn_id;
    grouped_tile(xcd_contiguous_id(blockIdx.x, p.tiles_m * p.tiles_n), p.tiles_m, p.tiles_n, 4, tm_id, tn_id);
    const int m0 = (int)tm_id * BM, n0 = (int)tn_id * BN;

    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(A), 0, (int)((size_t)M * K * sizeof(float)), kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(B), 0, (int)((size_t)K * N * sizeof(float)), kBufferRsrcWord3);
    constexpr int kOut = 0x7ffffff0;  // past the end of any operand: the load returns 0

    const int k_begin = SPLIT ? (int)blockIdx.y * p.kchunk : 0;
    const int k_end = SPLIT ? min(K, k_begin + p.kchunk) : K;
    const int steps = (k_end - k_begin + BK - 1) / BK;
    const int iters = (steps + KG - 1) / KG;

    T t;
    t.clear();
    const int k0 = k_begin + t.grp * BK;
    if (t.stages_a()) {
        // (both operands contiguous along k: A is cleared past K)
        std::conditional_t<TA, ColLoader<BM, T::CA, KG>, RowLoader<BM, T::CA, KG, TB>> ld(ra, t.stager(), m0, TA ? M : K, k0);
        t.template run<true>(smem, ld, iters);
    } else {
        std::conditional_t<TB, RowLoader<BN, T::CB, KG, false>, ColLoader<BN, T::CB, KG>> ld(rb, t.stager(), n0, TB ? K : N, k0);
        t.template run<false>(smem, ld, iters);
    }
    t.reduce(smem);

    // where this lane's elements of C are: row of (block, register), column of block
    auto row_of = [&](int q) { return TA && T::CA == 2 ? pair_slot(q) : q; };
    const int mw = m0 + t.row0();
    const int cb = n0 + t.wn * WN + (!TB && T::CB == 2 ? pair_slot(t.lr) : t.lr);

    // sums that are not all finite are recomputed in fp32 (split.hpp)
    if (t.not_finite()) {
        // four k of a row whose k are contiguous, or of a k-major operand's column
        auto along = [&](__amdgpu_buffer_rsrc_t r, bool in, int row, int k) {
            f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, pick(in, (row * K + k) * 4, kOut), 0, 0));
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = k + q < k_end ? v[q] : 0.0f;
            return v;
        };
        auto across = [&](__amdgpu_buffer_rsrc_t r, bool in, int col, int cols, int k) {
            f32x4 v;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     r, pick(in & (k + q < k_end), ((k + q) * cols + col) * 4, kOut), 0, 0));
            return v;
        };
        t.recompute(
            k_begin, k_end,
            [&](int i, int k) {
                const int row = mw + 32 * i + row_of(t.lr);
                return TA ? across(ra, row < M, row, M, k) : along(ra, row < M, row, k);
            },
            [&](int j, int k) {
                const int col = cb + 32 * j;
                return TB ? along(rb, col < N, col, k) : across(rb, col < N, col, N, k);
            });
    }

    // C through a buffer resource: rows past M fall past its end and columns
    // past N are sent there, so an edge tile takes the same straight code (a
    // launch of few tiles pays for every line of code it fetches: with
    // per-element checks 128 x 128 tiles started in 16 us instead of 7).
    float* const out = SPLIT ? p.ws + ((size_t)g * p.splits + blockIdx.y) * (size_t)M * N : C;
    const int c_bytes = (int)((size_t)M * N * sizeof(float));
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(out, 0, c_bytes, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(R), 0, R && !SPLIT ? c_bytes : 0, kBufferRsrcWord3);
    const float* __restrict__ bias = SPLIT ? nullptr : p.bias[g];
    float bv[TN];
    int co[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = cb + 32 * j;
        bv[j] = bias && col < N ? bias[col] : 0.0f;
        co[j] = pick(col < N, ((mw + (TA && T::CA == 2 ? 8 : 4) * t.lk) * N + col) * 4, kOut);
    }
    // row_of(8 (r / 4) + 4 lk + r % 4) less its lane part (4 lk, twice that in pairs)
    auto row_off = [&](int i, int r) { return (32 * i + row_of(8 * (r >> 2) + (r & 3))) * N * 4; };
    with_act(SPLIT ? (int)kActNone : p.act, [&](auto act_c) {
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (int i = 0; i < T::TS; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x16 rv = {};
                if (!SPLIT && R) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        rv[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rr, co[j], row_off(i, r), 0));
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float v = act_fixed<ACT>(t.acc[i][j][r] + bv[j]);
                    const float w = !SPLIT && R ? v + rv[r] : v;
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, w), rc, co[j], row_off(i, r), 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    });
}

template <int BM, int BN, int WM, int WN, int KG, bool SPLIT, int MODE, int SCHED>
void launch(hipStream_t stream, GemmParams& p, int count, bool ta, bool tb) {
    p.tiles_m = (uint32_t)((p.M + BM - 1) / BM);
    p.tiles_n = (uint32_t)((p.N + BN - 1) / BN);
    const dim3 grid(p.tiles_m * p.tiles_n, (unsigned)p.splits, (unsigned)count);
    const dim3 block(64 * (BM / WM) * (BN / WN) * KG);
    if (ta)
        hipLaunchKernelGGL((gemm_f32_split<BM, BN, WM, WN, KG, true, false, SPLIT, MODE, SCHED>), grid, block, 0, stream, p);
    else if (tb)
        hipLaunchKernelGGL((gemm_f32_split<BM, BN, WM, WN, KG, false, true, SPLIT, MODE, SCHED>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((gemm_f32_split<BM, BN, WM, WN, KG, false, false, SPLIT, MODE, SCHED>), grid, block, 0, stream, p);
}

}  // namespace

int launch_gemm_split(lancius_hip_ctx* ctx, GemmParams& p, int count, bool ta, bool tb, int tile) {
    const char* name = "gemm_f32_split 128x128";
    if (tile == kSplit256) {
        name = "gemm_f32_split 256x256";
        launch<256, 256, 64, 128, 1, false, kOneSum, 5>(ctx->stream, p, count, ta, tb);
    } else if (tile == kSplit256x128) {
        name = "gemm_f32_split 256x128";
        launch<256, 128, 64, 64, 1, false, kTwoSums, 0>(ctx->stream, p, count, ta, tb);
    } else if (p.splits == 1) {
        launch<128, 128, 64, 64, 2, false, kTwoSums, 5>(ctx->stream, p, count, ta, tb);
    } else {
        name = "gemm_f32_split 128x128 split K";
        launch<128, 128, 64, 64, 2, true, kTwoSums, 5>(ctx->stream, p, count, ta, tb);
    }
    return check_launch(name);
}

}  // namespace lancius
