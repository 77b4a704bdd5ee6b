// The k loop of a tile of split products (split.hpp): what the GEMM, the
// convolution and its weight gradient share.  A loader per operand brings the
// operand's values into registers in the order of MFMA operands.
//
// What bounds it: the matrix cores, at the clock the power limit leaves them
// (dense bf16 products alone run at 1.76 PFLOP/s on this card, 293 TFLOP/s of
// split products).  So the design spends as little as it can beside them:
//  * Each operand element is loaded and split once per workgroup (half the
//    waves stage A, half stage B: one of each on every SIMD) and read from
//    LDS as whole 16-byte MFMA operands: per part, chunk (k half, row) at
//    16 (row + rows k half), so reads and writes walk contiguous 512-byte
//    runs.
//  * Three LDS buffers and one barrier a step, three quarters (or half) into
//    the MFMAs: the next step's tile is split and written during the step's
//    first half while its successor's loads are in flight, and the first
//    operand reads of a step follow no barrier.  (Loads two steps ahead
//    measured no faster, and spilled.)
// MODE kOneSum adds all six products to one accumulator: 12 roundings per 16
// k at its magnitude against the 16 of v_mfma_f32_32x32x2_f32 (measured
// normwise error of a 4096^3 product: 1.02e-6, fp32 instructions 1.15e-6).
// MODE kTwoSums keeps the five small products apart until the end, 2 roundings
// per 16 k (4.0e-7), for twice the accumulators.
#pragma once

#include "split.hpp"

namespace lancius {

enum : int { kOneSum = 1, kTwoSums = 2 };

// Slot s of a 32-row group filled by row pairs (even rows first) -> row.
__device__ __forceinline__ int pair_slot(int s) { return s < 16 ? 2 * s : 2 * s - 31; }

// BM x BN tile, WM x WN per wave, KG k-groups of (BM/WM)(BN/WN) waves that
// take every KG-th k-step of 16.
template <int BM_, int BN_, int WM_, int WN_, int KG_, int MODE_, int SCHED_>
struct SplitTile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, KG = KG_, MODE = MODE_, SCHED = SCHED_;
    static constexpr int GW = (BM / WM) * (BN / WN);  // waves of a k-group
    static constexpr int GT = 64 * GW, NT = GT * KG;
    static constexpr int TM = WM / 32, TN = WN / 32;
    static constexpr int BK = 16, NBUF = 3;
    // chunks (8 k of a row) a thread stages: half the waves A, half B
    static constexpr int CA = 4 * BM / GT, CB = 4 * BN / GT;
    static_assert(CA >= 1 && CA <= 2 && CB >= 1 && CB <= 2 && CA * GT == 4 * BM && CB * GT == 4 * BN, "one or two");
    static constexpr int PLA = 2 * BM * 16, PLB = 2 * BN * 16;  // one part of one operand
    static constexpr int A_BYTES = 3 * PLA, BUF = A_BYTES + 3 * PLB;
    static constexpr int STAGE = KG * NBUF * BUF, RED = KG > 1 ? BM * BN * 4 : 0;
    static constexpr int SMEM = STAGE > RED ? STAGE : RED;
    static_assert(KG == 1 || (KG == 2 && TM == 2), "two k-groups exchange halves");
    static constexpr int TS = TM / KG;  // block rows a wave keeps after reduce()
    static constexpr int TML = MODE == kTwoSums ? TM : 1, TNL = MODE == kTwoSums ? TN : 1;

    f32x16 acc[TM][TN], low[TML][TNL];
    int grp, gw, lane, lr, lk, wm, wn;

    __device__ __forceinline__ SplitTile() {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lane = threadIdx.x & 63;
        grp = KG > 1 ? wave / GW : 0;
        gw = wave % GW;
        wm = gw / (BN / WN);
        wn = gw % (BN / WN);
        lr = lane & 31;
        lk = lane >> 5;
    }
    __device__ __forceinline__ bool stages_a() const { return gw < GW / 2; }
    __device__ __forceinline__ int stager() const { return (gw % (GW / 2)) * 64 + lane; }  // thread of its half

    static __device__ __forceinline__ SplitOperand get(const char* at, int pl) {
        SplitOperand s;
        s.h = *(const bf16x8*)(at);
        s.m = *(const bf16x8*)(at + pl);
        s.l = *(const bf16x8*)(at + 2 * pl);
        return s;
    }

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};
#pragma unroll
        for (int i = 0; i < TML; ++i)
#pragma unroll
            for (int j = 0; j < TNL; ++j) low[i][j] = f32x16{};
    }

    // Adds `iters` steps.  L stages one operand: load() brings the next of
    // this k-group's steps into registers, chunk(c) is its c-th chunk and
    // wr[c] that chunk's place in a buffer.  Every wave of the workgroup calls
    // this the same number of steps, IS_A in the waves of stages_a().
    template <bool IS_A, class L>
    __device__ __forceinline__ void run(char* smem, L& ld, int iters) {
        constexpr int CN = IS_A ? CA : CB, PL = IS_A ? PLA : PLB;
        char* const base = smem + grp * NBUF * BUF;
        const int a_rd = (lk * BM + wm * WM + lr) * 16;
        const int b_rd = A_BYTES + (lk * BN + wn * WN + lr) * 16;
        auto stage = [&](int buf, int c) {
            if (c >= CN) return;
            const SplitOperand s = split8_up(ld.chunk(c));
            char* const at = base + buf + (IS_A ? 0 : A_BYTES) + ld.wr[c < CN ? c : 0];
            *(bf16x8*)(at) = s.h;
            *(bf16x8*)(at + PL) = s.m;
            *(bf16x8*)(at + 2 * PL) = s.l;
        };
        ld.load();
        stage(0, 0);
        stage(0, 1);
        ld.load();
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
                if (j == 0) stage(nxt, 0);
                if (j == (TN == 4 ? 1 : 0)) {
                    stage(nxt, 1);
                    ld.load();
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
    }

    // The whole sums, after run() and a settle, as the operands have them.  Two k-groups: each keeps half
    // of the wave's block rows (acc[0 .. TS), rows wm WM + 32 grp ..) and adds
    // the other group's sums of them (a + b is the same either way round, so
    // results do not depend on which group ends first).
    __device__ __forceinline__ void reduce(char* smem) {
        settle(acc);
        if constexpr (MODE == kTwoSums) {
            settle(low);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] *= kSplitDown;
        if constexpr (KG > 1) {
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
                for (int r = 0; r < 16; ++r)
                    acc[0][j][r] = (grp ? acc[1][j][r] : acc[0][j][r]) + red[at(1 - grp, j, r)];
        }
    }
    // the wave's first block row of those it keeps
    __device__ __forceinline__ int row0() const { return wm * WM + 32 * (KG > 1 ? grp : 0); }

    // Some kept sum is not finite (an infinite or NaN input, or a value or
    // product beyond the scaled range): the wave recomputes its blocks in fp32.
    __device__ __forceinline__ bool not_finite() const {
        float none = 0.0f, probe = 0.0f;
        asm("" : "+v"(none));  // a register: the compiler may not fold x * 0
#pragma unroll
        for (int i = 0; i < TS; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) probe = fmaf(acc[i][j][r], none, probe);
        return __any(!(probe == 0.0f));
    }

    // The wave's kept blocks with the fp32 instructions, over k in [k_begin,
    // k_end): a(i, k) and b(j, k) give k .. k + 3 of this lane's row of block
    // row i and column of block column j, 0 from k_end on.  A group of 8 k is
    // loaded while the one before it is multiplied, and an operand serves
    // every block of its row or column.  Bound by the fp32 matrix rate: with a
    // NaN in each row 4096^3 takes 1777 us (585 without; block by block, two k
    // at a time, 5518; fp32 kernels alone 1037), N32 64->128 3x3 56^2 310 (113;
    // 904; 151), its weight gradient 315 (110; 747; 167).
    template <class FA, class FB>
    __device__ __forceinline__ void recompute(int k_begin, int k_end, const FA& a, const FB& b) {
        f32x4 av[2][TS], bv[2][TN];
#pragma unroll
        for (int i = 0; i < TS; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x16{};
        auto load = [&](int s, int k) {
#pragma unroll
            for (int i = 0; i < TS; ++i) av[s][i] = a(i, k + 4 * lk);
#pragma unroll
            for (int j = 0; j < TN; ++j) bv[s][j] = b(j, k + 4 * lk);
        };
        auto multiply = [&](int s) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < TS; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[s][i][q], bv[s][j][q], acc[i][j], 0, 0, 0);
        };
        load(0, k_begin);
#pragma unroll 1
        for (int k = k_begin; k < k_end; k += 16) {
            load(1, k + 8);
            multiply(0);
            load(0, k + 16);
            multiply(1);
        }
        settle(acc);
    }
};

// Loaders of a matrix through a buffer resource: rows past it and k-major rows
// past K read 0; past K of a row that runs along k lie the next row's values,
// which the other operand's zeros cancel.  No alignment is asked for.

// [rows][K], k contiguous: a thread takes 32 bytes (8 k) of one row, or of
// two BE/2 apart.  MASK: clear values past K.
template <int BE, int CN, int KG, bool MASK>
struct RowLoader {
    __amdgpu_buffer_rsrc_t rs;
    int wr[CN], off[CN], k_next, kh, K;
    f32x8 s[CN];
    __device__ __forceinline__ RowLoader(__amdgpu_buffer_rsrc_t rs_, int st, int e0, int K_, int k0) : rs(rs_), K(K_) {
        kh = (st >> 5) & 1;
        const int row = (st & 31) + 32 * (st >> 6);
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            wr[c] = (kh * BE + row + c * (BE / 2)) * 16;
            off[c] = ((e0 + row + c * (BE / 2)) * K + 8 * kh) * 4;
        }
        k_next = k0;
    }
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off[c], k_next * 4, 0));
            const f32x4 y = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off[c] + 16, k_next * 4, 0));
            s[c] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        k_next += 16 * KG;
    }
    __device__ __forceinline__ f32x8 chunk(int c) const {
        f32x8 x = s[c];
        if constexpr (MASK) {
            const int left = K - (k_next - 16 * KG) - 8 * kh;
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = i < left ? x[i] : 0.0f;
        }
        return x;
    }
};

// [K][cols], k-major: a thread takes a column, or a pair of columns, over 8 k;
// the transposition is the choice of registers.  Pairs fill the slots even
// columns first (pair_slot).
template <int BE, int CN, int KG>
struct ColLoader {
    __amdgpu_buffer_rsrc_t rs;
    int wr[CN], off, k_next, cols;
    f32x8 s[CN];
    __device__ __forceinline__ ColLoader(__amdgpu_buffer_rsrc_t rs_, int st, int e0, int cols_, int k0)
        : rs(rs_), cols(cols_) {
        const int kh = st / (BE / CN), cj = st % (BE / CN);
        const int slot = CN == 2 ? (cj / 16) * 32 + (cj % 16) : cj;
#pragma unroll
        for (int c = 0; c < CN; ++c) wr[c] = (kh * BE + slot + 16 * c) * 16;
        off = (8 * kh * cols + e0 + CN * cj) * 4;
        k_next = k0;
    }
    __device__ __forceinline__ void load() {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int so = (k_next + i) * cols * 4;
            if constexpr (CN == 2) {
                const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, so, 0));
                s[0][i] = v.x;
                s[CN - 1][i] = v.y;
            } else {
                s[0][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, so, 0));
            }
        }
        k_next += 16 * KG;
    }
    __device__ __forceinline__ f32x8 chunk(int c) const { return s[c]; }
};

}  // namespace lancius
