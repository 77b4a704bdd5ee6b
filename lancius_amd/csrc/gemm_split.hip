// fp32 GEMM on the bf16 matrix cores: both operands are split into three bf16
// parts on the way into LDS and multiplied as six bf16 products (split.hpp).
#include "gemm.hpp"
#include "split.hpp"

namespace lancius {
namespace {

// Slot s of a 32-row group filled by column pairs (even columns first) -> column.
__device__ __forceinline__ int pair_slot(int s) { return s < 16 ? 2 * s : 2 * s - 31; }

// One BM x BN tile of C per workgroup, WM x WN per wave, KG k-groups of
// (BM/WM)(BN/WN) waves that take every KG-th k-step of 16 and add their sums
// through LDS at the end.
//
// What bounds it: the matrix cores, at the clock the power limit leaves them
// (dense bf16 products alone run at 1.76 PFLOP/s on this card, 293 TFLOP/s of
// split products).  So the design spends as little as it can beside them:
//  * Each operand element is loaded and split once per workgroup (half the
//    waves stage A, half stage B: one of each on every SIMD) and read from
//    LDS as whole 16-byte MFMA operands: per part, chunk (k half, row) at
//    16 (row + rows k half), so reads and writes walk contiguous 512-byte
//    runs.  An operand whose rows run along k is loaded as 32 bytes of one
//    row; one stored k-major as column pairs over 8 k, the transposition
//    being the choice of registers.  Pairs fill the slots even columns first
//    (pair_slot), which C's store undoes.
//  * Loads go through buffer resources: rows past the operand and k-major rows
//    past K read 0.  Past K of a row-contiguous operand lie the next row's
//    values, which the other operand's zeros cancel; when both are
//    row-contiguous (MASK), A is cleared.  No alignment is asked for.
//  * Three LDS buffers and one barrier a step, three quarters (or half) into
//    the MFMAs: the next step's tile is split and written during the step's
//    first half while its successor's loads are in flight, and the first
//    operand reads of a step follow no barrier.
// MODE kOneSum adds all six products to one accumulator: 12 roundings per 16
// k at its magnitude against the 16 of v_mfma_f32_32x32x2_f32 (measured
// normwise error at K = 4096: 1.02e-6, fp32 instructions 1.15e-6).  MODE
// kTwoSums keeps the five small products apart until the end, 2 roundings
// per 16 k (4.0e-7), for twice the accumulators.
enum : int { kOneSum = 1, kTwoSums = 2 };

template <int BM, int BN, int WM, int WN, int KG, bool TA, bool TB, bool SPLIT, int MODE, int SCHED>
__global__ void __launch_bounds__(64 * (BM / WM) * (BN / WN) * KG, 2) gemm_f32_split(const GemmParams p) {
    constexpr int GT = 64 * (BM / WM) * (BN / WN);  // threads of a k-group
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int BK = 16, NBUF = 3;
    constexpr int CH = 8;  // k per chunk: one lane's MFMA operand, 16 bytes a part
    constexpr int CA = 4 * BM / GT, CB = 4 * BN / GT;  // chunks a thread stages: half the waves A, half B
    static_assert(CA >= 1 && CA <= 2 && CB >= 1 && CB <= 2 && CA * GT == 4 * BM && CB * GT == 4 * BN, "one or two");
    constexpr int A_BYTES = 3 * 2 * BM * 16, B_BYTES = 3 * 2 * BN * 16;
    constexpr int BUF = A_BYTES + B_BYTES;
    constexpr int STAGE = KG * NBUF * BUF;
    constexpr int RED = KG > 1 ? BM * BN * 4 : 0;
    __shared__ __attribute__((aligned(16))) char smem[STAGE > RED ? STAGE : RED];

    const int g = blockIdx.z;
    const float* __restrict__ A = p.A[g];
    const float* __restrict__ B = p.B[g];
    float* __restrict__ C = p.C[g];
    const float* __restrict__ R = p.R[g];
    const int M = p.M, N = p.N, K = p.K;
    uint32_t tm_id, tn_id;
    grouped_tile(xcd_contiguous_id(blockIdx.x, p.tiles_m * p.tiles_n), p.tiles_m, p.tiles_n, 4, tm_id, tn_id);
    const int m0 = (int)tm_id * BM, n0 = (int)tn_id * BN;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    constexpr int GW = GT / 64;
    const int grp = KG > 1 ? wave / GW : 0, gw = wave % GW;
    const int wm = gw / (BN / WN), wn = gw % (BN / WN);
    const int lr = lane & 31, lk = lane >> 5;

    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(A), 0, (int)((size_t)M * K * sizeof(float)), kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(B), 0, (int)((size_t)K * N * sizeof(float)), kBufferRsrcWord3);
    constexpr int kOut = 0x7ffffff0;  // past the end of any operand: the load returns 0
    constexpr int PLA = 2 * BM * 16, PLB = 2 * BN * 16;  // one part of one operand
    char* const base = smem + grp * NBUF * BUF;
    const int a_rd = (lk * BM + wm * WM + lr) * 16;
    const int b_rd = A_BYTES + (lk * BN + wn * WN + lr) * 16;
    auto get = [&](const char* at, int pl) {
        SplitOperand s;
        s.h = *(const bf16x8*)(at);
        s.m = *(const bf16x8*)(at + pl);
        s.l = *(const bf16x8*)(at + 2 * pl);
        return s;
    };
    auto put = [&](char* at, int pl, const SplitOperand& s) {
        *(bf16x8*)(at) = s.h;
        *(bf16x8*)(at + pl) = s.m;
        *(bf16x8*)(at + 2 * pl) = s.l;
    };
    f32x16 low[MODE == kTwoSums ? TM : 1][MODE == kTwoSums ? TN : 1];
    if constexpr (MODE == kTwoSums) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) low[i][j] = f32x16{};
    }

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const int k_begin = SPLIT ? (int)blockIdx.y * p.kchunk : 0;
    const int k_end = SPLIT ? min(K, k_begin + p.kchunk) : K;
    const int steps = (k_end - k_begin + BK - 1) / BK;
    const int iters = (steps + KG - 1) / KG;

    auto k_loop = [&](auto role) {
        constexpr bool IS_A = decltype(role)::value;
        constexpr bool KC = IS_A ? !TA : TB;   // k contiguous in memory
        constexpr bool MASK = IS_A && !TA && TB;  // both operands k-contiguous: A is cleared past K
        const __amdgpu_buffer_rsrc_t rs = IS_A ? ra : rb;
        const int ext = IS_A ? M : N, e0 = IS_A ? m0 : n0;
        constexpr int BE = IS_A ? BM : BN, CN = IS_A ? CA : CB, PL = IS_A ? PLA : PLB;
        const int st = (gw % (GW / 2)) * 64 + lane;
        // k-contiguous: rows krow (and krow + BE/2), k half kh; otherwise
        // columns 2 cj, 2 cj + 1 (or column cj), k half kh
        const int kh = KC ? (st >> 5) & 1 : st / (BE / CN);
        const int krow = (st & 31) + 32 * (st >> 6), cj = st % (BE / CN);
        const int slot0 = KC ? krow : CN == 2 ? (cj / 16) * 32 + (cj % 16) : cj;
        const int slot1 = KC ? krow + BE / 2 : slot0 + 16;
        const int wr0 = (IS_A ? 0 : A_BYTES) + (kh * BE + slot0) * 16;
        const int wr1 = (IS_A ? 0 : A_BYTES) + (kh * BE + slot1) * 16;
        const int voff0 = KC ? ((e0 + krow) * K + CH * kh) * 4 : (CH * kh * ext + e0 + CN * cj) * 4;
        const int voff1 = voff0 + (BE / 2) * K * 4;  // KC only
        struct Staged {
            f32x8 c[CN];
        };
        int k_next = k_begin + grp * BK;
        auto load_tile = [&](Staged& s) {
            if constexpr (KC) {
                const int so = k_next * 4;
#pragma unroll
                for (int c = 0; c < CN; ++c) {
                    const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, c ? voff1 : voff0, so, 0));
                    const f32x4 y = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (c ? voff1 : voff0) + 16, so, 0));
                    s.c[c] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int so = (k_next + i) * ext * 4;
                    if constexpr (CN == 2) {
                        const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, voff0, so, 0));
                        s.c[0][i] = v.x;
                        s.c[1][i] = v.y;
                    } else {
                        s.c[0][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, voff0, so, 0));
                    }
                }
            }
            k_next += KG * BK;
        };
        auto stage = [&](const Staged& s, int buf, int c, int k0) {
            if (c >= CN) return;
            f32x8 x = s.c[c < CN ? c : 0];
            if constexpr (MASK) {
                const int left = K - k0 - CH * kh;
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = i < left ? x[i] : 0.0f;
            }
            put(base + buf + (c ? wr1 : wr0), PL, split8(x));
        };
        Staged s;
        load_tile(s);
        stage(s, 0, 0, k_next - KG * BK);
        stage(s, 0, 1, k_next - KG * BK);
        load_tile(s);
        __syncthreads();
        int cur = 0;
        for (int it = 0; it < iters; ++it) {
            const int nxt = cur + BUF == NBUF * BUF ? 0 : cur + BUF;
            SplitOperand a[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = get(base + cur + a_rd + i * 32 * 16, PLA);
            SplitOperand b = get(base + cur + b_rd, PLB);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                SplitOperand bn = b;
                if (j + 1 < TN) bn = get(base + cur + b_rd + (j + 1) * 32 * 16, PLB);
                f32x16 t[TM];
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = MODE == kOneSum ? acc[i][j] : low[i][j];
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].l, b.h, t[i]);
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].h, b.l, t[i]);
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].m, b.m, t[i]);
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].m, b.h, t[i]);
#pragma unroll
                for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].h, b.m, t[i]);
                if constexpr (MODE == kTwoSums) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) low[i][j] = t[i];
#pragma unroll
                    for (int i = 0; i < TM; ++i) acc[i][j] = mfma_bf16(a[i].h, b.h, acc[i][j]);
                } else {
#pragma unroll
                    for (int i = 0; i < TM; ++i) t[i] = mfma_bf16(a[i].h, b.h, t[i]);
#pragma unroll
                    for (int i = 0; i < TM; ++i) acc[i][j] = t[i];
                }
                b = bn;
                if (j == 0) stage(s, nxt, 0, k_next - KG * BK);
                if (j == (TN == 4 ? 1 : 0)) {
                    stage(s, nxt, 1, k_next - KG * BK);
                    load_tile(s);
                }
                if (SCHED) {
#pragma unroll
                    for (int q = 0; q < 6 * TM; ++q) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, SCHED, 0);
                    }
                }
                if (j == (TN == 4 ? 2 : 0)) __syncthreads();
            }
            cur = nxt;
        }
    };
    if (gw < GW / 2)
        k_loop(std::integral_constant<bool, true>{});
    else
        k_loop(std::integral_constant<bool, false>{});
    settle(acc);
    if constexpr (MODE == kTwoSums) {
        settle(low);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
    }

    // Two k-groups: each keeps half of the wave's block rows, adds the other
    // group's sums of them (a + b is the same either way round, so results do
    // not depend on which group ends first) and stores that half.
    constexpr int TS = TM / KG;  // block rows a wave stores
    if constexpr (KG > 1) {
        static_assert(KG == 2 && TM == 2, "two k-groups exchange halves");
        float* const red = (float*)smem;
        auto at = [&](int from, int j, int r) { return ((from * GW + gw) * TN + j) * 1024 + r * 64 + lane; };
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[at(grp, j, r)] = grp ? acc[0][j][r] : acc[1][j][r];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][j][r] = (grp ? acc[1][j][r] : acc[0][j][r]) + red[at(1 - grp, j, r)];
    }

    // where this lane's elements of C are: row of (block, register), column of block
    const int i0 = KG > 1 ? grp : 0;
    auto row_of = [&](int q) { return TA && CA == 2 ? pair_slot(q) : q; };
    const int mw = m0 + wm * WM + 32 * i0;
    const int cb = n0 + wn * WN + (!TB && CB == 2 ? pair_slot(lr) : lr);

    // sums that are not all finite are recomputed in fp32 (split.hpp)
    float none = 0.0f, probe = 0.0f;
    asm("" : "+v"(none));  // a register: the compiler may not fold x * 0
#pragma unroll
    for (int i = 0; i < TS; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) probe = fmaf(acc[i][j][r], none, probe);
    if (__any(probe != 0.0f)) {
#pragma unroll
        for (int i = 0; i < TS; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int row = mw + 32 * i + row_of(lr), col = cb + 32 * j;
                f32x16 s = {};
#pragma unroll 1
                for (int k0 = k_begin; k0 < k_end; k0 += 2) {
                    const int k = k0 + lk;
                    const int ao = pick(k < k_end && row < M, (TA ? k * M + row : row * K + k) * 4, kOut);
                    const int bo = pick(k < k_end && col < N, (TB ? col * K + k : k * N + col) * 4, kOut);
                    const float av = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, ao, 0, 0));
                    const float bv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, bo, 0, 0));
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, s, 0, 0, 0);
                }
                settle(s);
                acc[i][j] = s;
            }
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
        co[j] = pick(col < N, ((mw + (TA && CA == 2 ? 8 : 4) * lk) * N + col) * 4, kOut);
    }
    // row_of(8 (r / 4) + 4 lk + r % 4) less its lane part (4 lk, twice that in pairs)
    auto row_off = [&](int i, int r) { return (32 * i + row_of(8 * (r >> 2) + (r & 3))) * N * 4; };
    with_act(SPLIT ? (int)kActNone : p.act, [&](auto act_c) {
        constexpr int ACT = decltype(act_c)::value;
#pragma unroll
        for (int i = 0; i < TS; ++i)
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
                    const float v = act_fixed<ACT>(acc[i][j][r] + bv[j]);
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
    if (tile == kSplit256)
        launch<256, 256, 64, 128, 1, false, kOneSum, 5>(ctx->stream, p, count, ta, tb);
    else if (tile == kSplit256x128)
        launch<256, 128, 64, 64, 1, false, kTwoSums, 0>(ctx->stream, p, count, ta, tb);
    else if (p.splits == 1)
        launch<128, 128, 64, 64, 2, false, kTwoSums, 4>(ctx->stream, p, count, ta, tb);
    else
        launch<128, 128, 64, 64, 2, true, kTwoSums, 4>(ctx->stream, p, count, ta, tb);
    return check_launch("gemm_f32_split");
}

}  // namespace lancius
