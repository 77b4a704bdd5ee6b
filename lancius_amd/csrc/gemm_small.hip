// Small fp32 products: a 16 x 16 or 32 x 32 tile of C per workgroup, K spread
// over its waves, one launch.
//
// Such a product is bound by latency, not by bytes or operations: the tiled
// kernels stage through LDS with a barrier a k-tile and give 64 x 64 tiles,
// so few CUs work, or they split K over workgroups and add the parts in a
// second launch or behind arrival counters.  Here each wave loads its K range
// straight into the matrix cores' operand registers, the next group of k
// while one is multiplied, and the waves' sums are added once through LDS in
// wave order.  The small tile is for latency: a workgroup's loads, mostly
// from beyond its own L2, cost more than its products (64 x 784 x 128: 32 x
// 32 tiles 6.5 us, 16 x 16 4.4, of which 4.2 are the launch).  Two groups
// more in flight measured the same or slower (more code to fetch).
//
// us a call, before and now: 64 x 784 x 128 10.3, 4.4; its input gradient
// 7.8, 4.2; 32 x 2048 x 128 9.4, 7.0; 512^3 11.9, 5.5.
#include <algorithm>
#include <cmath>

#include "gemm.hpp"

namespace lancius {
namespace {

// Operand fragments: four consecutive k of a row or column, a lane's share of
// a group.  KC: k is the contiguous axis (one 16-byte load).
template <bool KC>
__device__ __forceinline__ f32x4 fragment(__amdgpu_buffer_rsrc_t r, int off, int ld4) {
    if constexpr (KC) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    } else {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, j * ld4, 0));
        return v;
    }
}

template <int T, bool TA, bool TB, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) gemm_f32_small(const GemmParams p) {
    constexpr int NQ = T * T / 64;    // sums a lane holds
    constexpr int KS = 4 * (64 / T);  // k of a group: four MFMAs
    constexpr int NACC = T == 32 ? 2 : 4;  // (four of 16 registers halve the workgroups a CU holds)
    __shared__ float red[WAVES][NQ][64];
    const int g = blockIdx.z, M = p.M, N = p.N, K = p.K;
    const int lane = threadIdx.x & 63, lr = lane % T, lk = lane / T;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int m0 = (int)(blockIdx.x % p.tiles_m) * T, n0 = (int)(blockIdx.x / p.tiles_m) * T;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.A[g]), 0, (int)((size_t)M * K * sizeof(float)), kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.B[g]), 0, (int)((size_t)K * N * sizeof(float)), kBufferRsrcWord3);

    // this wave's groups [gi, ge) of KS k
    const int groups = (K + KS - 1) / KS, per = (groups + WAVES - 1) / WAVES;
    int gi = wave * per;
    const int ge = min(groups, gi + per);
    const int row = m0 + lr, col = n0 + lr;
    auto a_off = [&](int k) { return (TA ? k * M + row : row * K + k) * 4; };
    auto b_off = [&](int k) { return (TB ? col * K + k : k * N + col) * 4; };

    typedef float acc_t __attribute__((ext_vector_type(NQ)));
    f32x4 a[2], b[2];
    acc_t acc[NACC] = {};  // by k modulo NACC: short chains, and no MFMA waits for the one before
    auto load = [&](int s, int gl) {
        const int k = gl * KS + 4 * lk;
        a[s] = fragment<!TA>(ra, a_off(k), M * 4);
        b[s] = fragment<TB>(rb, b_off(k), N * 4);
    };
    auto multiply = [&](int s, int gl) {
        // (k-major operands end at K; the others run into their next row)
        if ((!TA || TB) && (gl + 1) * KS > K) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = gl * KS + 4 * lk + j < K;
                if (!TA) a[s][j] = in ? a[s][j] : 0.0f;
                if (TB) b[s][j] = in ? b[s][j] : 0.0f;
            }
        }
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
        load(0, gi);
        for (; gi + 2 < ge; gi += 2) {
            load(1, gi + 1);
            multiply(0, gi);
            load(0, gi + 2);
            multiply(1, gi + 1);
        }
        if (gi + 1 < ge) {
            load(1, gi + 1);
            multiply(0, gi);
            multiply(1, gi + 1);
        } else {
            multiply(0, gi);
        }
    }

    // C element (q, lane): column lane % T, row 8 (q / 4) + 4 (lane / T) + q % 4
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        float s = acc[0][q] + acc[1][q];
        if constexpr (NACC == 4) s += acc[2][q] + acc[3][q];
        red[wave][q][lane] = s;
    }
    __syncthreads();
    const float* __restrict__ bias = p.bias[g];
    const float* __restrict__ R = p.R[g];
#pragma unroll
    for (int q0 = 0; q0 < NQ; q0 += WAVES) {
        const int q = q0 + wave, r = m0 + 8 * (q >> 2) + 4 * lk + (q & 3);
        if (q < NQ && r < M && col < N) {
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) s += red[w][q][lane];
            if (bias) s += bias[col];
            s = apply_act(s, p.act);
            if (R) s += R[(size_t)r * N + col];
            p.C[g][(size_t)r * N + col] = s;
        }
    }
}

template <int T, int WAVES>
int launch(hipStream_t stream, GemmParams& p, int count, bool ta, bool tb) {
    p.tiles_m = (uint32_t)((p.M + T - 1) / T);
    p.tiles_n = (uint32_t)((p.N + T - 1) / T);
    const dim3 grid(p.tiles_m * p.tiles_n, 1, (unsigned)count), block(64 * WAVES);
    if (ta && tb)
        hipLaunchKernelGGL((gemm_f32_small<T, true, true, WAVES>), grid, block, 0, stream, p);
    else if (ta)
        hipLaunchKernelGGL((gemm_f32_small<T, true, false, WAVES>), grid, block, 0, stream, p);
    else if (tb)
        hipLaunchKernelGGL((gemm_f32_small<T, false, true, WAVES>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((gemm_f32_small<T, false, false, WAVES>), grid, block, 0, stream, p);
    return check_launch(LANCIUS_KERNEL_NAME("gemm_f32_small %dx%d x%d", T, T, WAVES));
}

}  // namespace

// Chosen from what a call costs (us; fitted to 400 products up to 2048 x 4096
// x 2048): its latency, which grows with K, and the operand bytes that the
// tiles read, which double the small tile's; rows loaded along k (TB) in short
// pieces cost more.  Against the other kernels (gemm_plan, skinny_us) 512 x
// 512 x 512 is 11.9 -> 5.5, 1024^3 stays (20.6; here 26).  A tile costs some
// time at any K (1920 x 78 x 1492: 18.5 staged, 24 here).
SmallPlan gemm_small_plan(size_t count, size_t M, size_t K, size_t N, bool tb) {
    const double k = (double)K;
    auto tiles = [&](size_t t) { return (double)(count * ((M + t - 1) / t) * ((N + t - 1) / t)); };
    if (M >= (1u << 24) || N >= (1u << 24)) return {16, 1e30};
    // (a long chain of groups of few tiles: 2 x 4096 x 32 transposed 15 us, 13 elsewhere)
    const double latency = 0.0017 * k + 0.0035 * std::max(0.0, k - 2048);
    const double us16 = 4.0 + latency + tiles(16) * (0.6e-3 + k * (tb ? 1.2e-5 : 0.9e-5));
    double t32 = tiles(32);
    if (K >= 512 && t32 > 256) t32 = 256 * std::ceil(t32 / 256);  // 16 waves: one tile a CU (270 tiles: 31 us, 216: 13)
    const double us32 = 4.0 + 2 * latency + t32 * (2e-3 + k * (tb ? 4.2e-5 : 2.2e-5));
    return us16 <= us32 ? SmallPlan{16, us16} : SmallPlan{32, us32};
}

int launch_gemm_small(lancius_hip_ctx* ctx, GemmParams& p, int count, bool ta, bool tb, int tile) {
    // 16 waves at a long K are for the sums: chains no longer than before
    if (tile == 32) return p.K < 512 ? launch<32, 8>(ctx->stream, p, count, ta, tb) : launch<32, 16>(ctx->stream, p, count, ta, tb);
    return p.K < 1024 ? launch<16, 8>(ctx->stream, p, count, ta, tb) : launch<16, 16>(ctx->stream, p, count, ta, tb);
}

}  // namespace lancius
