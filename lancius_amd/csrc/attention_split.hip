// Attention on the bf16 matrix cores: the fp32 kernel's transposed formulation
// (attention.hip) with K, Q, V and the probabilities split into three bf16
// parts each and multiplied as six products (split.hpp).
#include "attention.hpp"
#include "split.hpp"

namespace lancius {
namespace {

typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

constexpr int kQueries = 128;  // per workgroup, 32 per wave
constexpr int kKeys = 32;      // per step

// The scaled range (split.hpp) here: V is scaled as there.  Q (times the score
// scale) carries 2^32: past 2^96 it overflows and is recomputed, so what a key
// below 2^-110 loses, 2^-134, stays under 2^-31 in a score, whose absolute
// error counts, and K needs no scale.  Nor have probabilities one: below
// 2^-110 they keep 8 to 16 bits, an error of 2^-134 of the largest.
constexpr float kQueryUp = 0x1p32f;

// D = head dim; KS = 2: eight waves, the second four taking the odd key
// blocks of the same queries (grids of at most one tile per CU).
//
// What bounds it: at D = 64 the matrix cores' 48 products a step and the 230
// vector instructions of the softmax, the splits of P and of the staged keys
// (B8 H16 S=2048 causal: matrix cores busy 0.52, vector unit 0.56 of the busy
// CUs' cycles); at D = 128 the products that wait for the softmax (busy 0.57,
// vector unit 0.45 in a ragged causal prefill).
//  * S^T = K Q^T and O^T += V^T P^T with v_mfma_f32_32x32x16_bf16: a lane owns
//    one query in both, and its 16 scores, in register order, are the two P^T
//    operands of the block: keys 16 s + 8 (e / 4) + 4 half + e % 4 for element
//    e of step s.  V is staged in that key order.
//  * Q is split once into registers (at D = 128 its low parts go to LDS: with
//    them in registers 43 spill, B8 S=2048 1852 us against 1440).  Two waves
//    split each K block into LDS, two each V block, as 16-byte operands at
//    (chunk, row): contiguous writes and reads.  V's columns are taken NB at a
//    time, column NB j + e at row j of d-block e, so loads and the stores of O
//    are NB floats wide.
//  * One buffer each: V of a step is written while its scores are formed, the
//    next K after them.  For D < 128 the scores run a step ahead, so their
//    products overlap the softmax of the step before in the same wave (B4
//    S=1024 causal 75 -> 68 us; D = 128 has no registers for it).
//  * P V of a block is summed apart and added with the rescale of O in one
//    fused multiply-add: one rounding per 32 keys at O's magnitude (normwise
//    error at B8 S=2048 D = 64: fp32 instructions 6.6e-7, this 2.5e-7).
template <int D, int KS>
__global__ void __launch_bounds__(256 * KS, 2) attention_split(const AttnParams p) {
    constexpr int NB = D / 32;   // d-blocks of 32, floats of a V row per staging lane
    constexpr int QS = D / 16;   // MFMA steps over d
    constexpr int PART = kKeys * D * 2, BLOCK = 3 * PART;  // one part, one K or V block
    constexpr int GROUP = 2 * BLOCK;
    constexpr bool QL = D == 128;  // Q's low parts live in LDS
    constexpr bool PIPE = D < 128;
    constexpr int QLOW = QL ? kQueries * D * 2 : 0;
    constexpr int PER = 16 * NB + 2;                       // a lane's hand-off: O^T registers, m, l
    constexpr int RED = KS > 1 ? 4 * PER * 64 * 4 : 0;
    __shared__ __attribute__((aligned(16))) char smem[KS * GROUP + QLOW > RED ? KS * GROUP + QLOW : RED];

    // task order: see attention_mfma (attention.hip)
    const int hz = p.H * p.Z;
    const int task = (int)blockIdx.x;
    const int t_rank = task / hz;
    const int rem = task - t_rank * hz;
    const int z = rem / p.H;
    const int h = rem - z * p.H;
    const int g = z / p.batch, b = z % p.batch;
    const int half_t = p.q_tiles / 2;
    const int qt = !p.causal                                                ? t_rank
                   : (p.pair_tiles && t_rank >= p.q_tiles - half_t) ? t_rank - (p.q_tiles - half_t)
                                                                      : p.q_tiles - 1 - t_rank;
    const int S = p.S, H = p.H, Skv = p.Skv;
    const int off = Skv - S;
    const int hk = h / (H / p.Hkv);
    const size_t row_stride = (size_t)H * D;
    const int kv_stride = p.Hkv * D;
    const size_t base = ((size_t)b * S * H + h) * D;
    const size_t kv_base = ((size_t)b * Skv * p.Hkv + hk) * D;
    const float* __restrict__ Qg = p.Q[g] + base;
    const float* __restrict__ Kg = p.K[g] + kv_base;
    const float* __restrict__ Vg = p.V[g] + kv_base;
    float* __restrict__ Og = p.O[g] + base;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int grp = KS > 1 ? wave >> 2 : 0;
    const int gw = wave & 3;
    const int wq = grp ? 3 - gw : gw;  // long and short causal rows share a SIMD
    const int lq = lane & 31, lk = lane >> 5;
    const int q0 = qt * kQueries;
    const int qw0 = q0 + wq * 32;
    const int q = qw0 + lq;
    const bool q_valid = q < S;
    char* const kbase = smem + grp * GROUP;
    char* const vbase = kbase + BLOCK;
    char* const ql = smem + KS * GROUP + wq * (32 * D * 2) + lane * 16;

    const int kv_bytes = ((Skv - 1) * kv_stride + D) * (int)sizeof(float);
    const __amdgpu_buffer_rsrc_t kbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Kg), 0, kv_bytes, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t vbuf =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Vg), 0, kv_bytes, kBufferRsrcWord3);

    // Q^T operands: step s covers d = 16 s + 8 lk ..
    SplitOperand qf[QS];
    {
        const f32x4* src = (const f32x4*)(Qg + (size_t)(q_valid ? q : 0) * row_stride + 8 * lk);
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const f32x4 x = src[4 * s], y = src[4 * s + 1];
            f32x8 v = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
            v = v * (p.qscale * kQueryUp);
            qf[s] = split8(v);
            // (this lane's own slot: with two k-groups both write the same values)
            if constexpr (QL) *(bf16x8*)(ql + s * 1024) = qf[s].l;
        }
    }

    const int kv_end = p.causal ? max(0, min(Skv, q0 + kQueries + off)) : Skv;
    const int nblocks = (kv_end + kKeys - 1) / kKeys;
    const int nsteps = (nblocks + KS - 1) / KS;

    // Staging: waves 0, 1 of the group take K (key st % 32, NB chunks of 8 d),
    // waves 2, 3 take V (the keys of one MFMA operand chunk, NB columns).
    const bool is_k = gw < 2;
    const int st = (gw & 1) * 64 + lane;
    const int oct = st >> 5, sj = st & 31;
    int s_off, s_wr;
    if (is_k) {
        s_off = (sj * kv_stride + oct * NB * 8) * 4;
        s_wr = (oct * NB * 32 + sj) * 16;  // chunk c at 512 c + 16 key
    } else {
        // octet oct = 2 s + half: keys 16 s + 4 half + {0..3, 8..11}
        s_off = ((16 * (oct >> 1) + 4 * (oct & 1)) * kv_stride + sj * NB) * 4;
        s_wr = (oct * D + sj) * 16;        // column NB j + e at 16 (32 e + j) of the octet
    }
    f32x8 sreg[NB];
    auto load_block = [&](auto role, int blk) {  // this wave's share of key block blk (0 past the keys)
        const int so = s_off + blk * kKeys * kv_stride * 4;
        if constexpr (decltype(role)::value) {
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const f32x4 x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(kbuf, so + 32 * c, 0, 0));
                const f32x4 y = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(kbuf, so + 32 * c + 16, 0, 0));
                sreg[c] = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int ro = (8 * (i >> 2) + (i & 3)) * kv_stride * 4;
                if constexpr (NB == 1) {
                    sreg[0][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(vbuf, so, ro, 0));
                } else if constexpr (NB == 2) {
                    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(vbuf, so, ro, 0);
#pragma unroll
                    for (int e = 0; e < 2; ++e) sreg[e][i] = __builtin_bit_cast(float, (unsigned)v[e]);
                } else if constexpr (NB == 3) {
                    const u32x3 v = __builtin_amdgcn_raw_buffer_load_b96(vbuf, so, ro, 0);
#pragma unroll
                    for (int e = 0; e < 3; ++e) sreg[e][i] = __builtin_bit_cast(float, (unsigned)v[e]);
                } else {
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(vbuf, so, ro, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) sreg[e][i] = __builtin_bit_cast(float, (unsigned)v[e]);
                }
            }
        }
    };
    auto store_block = [&](auto role, char* to) {
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const SplitOperand s = decltype(role)::value ? split8(sreg[c]) : split8_up(sreg[c]);
            char* at = to + s_wr + c * 512;
            *(bf16x8*)at = s.h;
            *(bf16x8*)(at + PART) = s.m;
            *(bf16x8*)(at + 2 * PART) = s.l;
        }
    };
    auto get = [&](const char* at) {
        SplitOperand s;
        s.h = *(const bf16x8*)at;
        s.m = *(const bf16x8*)(at + PART);
        s.l = *(const bf16x8*)(at + 2 * PART);
        return s;
    };

    f32x16 o_acc[NB];  // O^T: block e, row j is d = NB j + e
#pragma unroll
    for (int e = 0; e < NB; ++e) o_acc[e] = f32x16{};
    float m_run = -1e30f;
    float l_part = 0.0f;

    // Register r of lane l holds key kb + 8*(r/4) + 4*(l/32) + r%4.
    auto mask = [&](f32x16& s, int kb) {
        if ((p.causal && kb + kKeys - 1 > qw0 + off) || kb + kKeys > Skv) {
            const int lim = min(Skv - 1, p.causal ? q + off : Skv - 1) - (kb + 4 * lk);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 8 * (r >> 2) + (r & 3) > lim ? -INFINITY : s[r];
        }
    };
    // Running maximum and sum; probabilities in place of the scores, which come
    // multiplied by 1 / down.  Returns the factor of the sums so far.
    auto softmax = [&](f32x16& s, float down) {
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, mx), __builtin_bit_cast(unsigned, mx),
                                                         false, false);  // the other half's maximum
        mx = fmaxf(__builtin_bit_cast(float, (unsigned)sw[0]), __builtin_bit_cast(float, (unsigned)sw[1]));
        const float m_new = fmaxf(m_run, mx * down);
        const float corr = exp2_raw(m_run - m_new);
        m_run = m_new;
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = exp2_raw(fmaf(s[r], down, -m_new));
            psum += s[r];
        }
        l_part = l_part * corr + psum;
        return corr;
    };
    auto scores = [&]() {  // S^T of the staged K block
        const char* kc = kbase + (lk * 32 + lq) * 16;
        f32x16 s0 = {}, s1 = {};
        // (the next step's operands are read before this step's MFMAs; the
        // scheduling barrier keeps more of them from being read ahead into
        // registers that are not there)
        SplitOperand k = get(kc);
        bf16x8 low = QL ? *(const bf16x8*)ql : qf[0].l;
#pragma unroll
        for (int s = 0; s < QS; ++s) {
            const SplitOperand kn = s + 1 < QS ? get(kc + (s + 1) * 1024) : k;
            const bf16x8 ln = s + 1 == QS ? low : QL ? *(const bf16x8*)(ql + (s + 1) * 1024) : qf[s + 1].l;
            f32x16& c = s & 1 ? s1 : s0;
            c = mfma_bf16(k.l, qf[s].h, c);
            c = mfma_bf16(k.h, low, c);
            c = mfma_bf16(k.m, qf[s].m, c);
            c = mfma_bf16(k.m, qf[s].h, c);
            c = mfma_bf16(k.h, qf[s].m, c);
            c = mfma_bf16(k.h, qf[s].h, c);
            k = kn;
            low = ln;
            if constexpr (!PIPE) __builtin_amdgcn_sched_barrier(0);
        }
        s0 += s1;
        pin(s0);  // read out of the matrix results in this block (split.hpp)
        return s0;
    };

    auto key_loop = [&](auto role) {
        constexpr bool IS_K = decltype(role)::value;
        f32x16 s_cur = {};
        load_block(role, grp);
        if (IS_K) {
            store_block(role, kbase);
            load_block(role, grp + KS);
        }
        __syncthreads();
        if constexpr (PIPE) {
            s_cur = scores();
            mask(s_cur, grp * kKeys);
            __syncthreads();
            if (IS_K) {
                store_block(role, kbase);
                load_block(role, grp + 2 * KS);
            }
            __syncthreads();
        }
        for (int it = 0; it < nsteps; ++it) {
            const int blk = it * KS + grp, kb = blk * kKeys;
            const bool active = blk < nblocks && (!p.causal || kb <= qw0 + 31 + off);
            f32x16 s_next = {};
            float corr = 1.0f;
            SplitOperand pf[2];
            if (active) {
                if constexpr (PIPE) {
                    s_next = scores();
                } else {
                    s_cur = scores();
                    mask(s_cur, kb);
                }
                corr = softmax(s_cur, 1.0f / kQueryUp);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    f32x8 x;
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = s_cur[8 * s + e];
                    pf[s] = split8(x);
                }
            }
            if (!IS_K) {  // every wave is past the last step's V
                store_block(role, vbase);
                load_block(role, blk + KS);
            }
            __syncthreads();
            if (IS_K) {  // every wave is past the staged K
                store_block(role, kbase);
                load_block(role, blk + (PIPE ? 3 : 2) * KS);
            }
            if (active) {
                SplitOperand v = get(vbase + (lk * D + lq) * 16);
#pragma unroll
                for (int e = 0; e < NB; ++e) {
                    f32x16 t = {};
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int n = 2 * e + s + 1;
                        const SplitOperand vn = n < 2 * NB ? get(vbase + ((2 * (n & 1) + lk) * D + 32 * (n >> 1) + lq) * 16) : v;
                        t = mfma_bf16(v.l, pf[s].h, t);
                        t = mfma_bf16(v.h, pf[s].l, t);
                        t = mfma_bf16(v.m, pf[s].m, t);
                        t = mfma_bf16(v.m, pf[s].h, t);
                        t = mfma_bf16(v.h, pf[s].m, t);
                        t = mfma_bf16(v.h, pf[s].h, t);
                        v = vn;
                        if constexpr (!PIPE) __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[e][r] = fmaf(o_acc[e][r], corr, t[r]);
                    pin(o_acc[e]);
                }
                if constexpr (PIPE) {
                    mask(s_next, kb + KS * kKeys);
                    s_cur = s_next;
                }
            }
            __syncthreads();
        }
    };
    if (nsteps > 0) {
        if (is_k)
            key_loop(std::integral_constant<bool, true>{});
        else
            key_loop(std::integral_constant<bool, false>{});
    }

    // Sums that are not all finite (infinite or NaN inputs, values or scores
    // beyond the scaled range): the wave's key blocks again with the fp32
    // instructions.  With a NaN in every sequence B8 H16 S=2048 D=64 causal
    // takes 1423 us (440 without; with operands loaded one at a time 2542; the
    // fp32 kernel alone 643), D=128 4998 (1765; 9497; 2285).
    float none = 0.0f, probe = l_part * 0.0f;
    asm("" : "+v"(none));
#pragma unroll
    for (int e = 0; e < NB; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(o_acc[e][r], none, probe);
    if (!__any(!(probe == 0.0f))) {
#pragma unroll
        for (int e = 0; e < NB; ++e) o_acc[e] *= 1.0f / kSplitUp;
    } else {
#pragma unroll
        for (int e = 0; e < NB; ++e) o_acc[e] = f32x16{};
        m_run = -1e30f;
        l_part = 0.0f;
        const float* qrow = Qg + (size_t)(q_valid ? q : 0) * row_stride;
#pragma unroll 1
        for (int it = 0; it < nsteps; ++it) {
            const int blk = it * KS + grp, kb = blk * kKeys;
            if (!(blk < nblocks && (!p.causal || kb <= qw0 + 31 + off))) continue;
            // (V's loads leave before the scores are formed, where there are
            // registers for them: with D = 128 the main loop would spill)
            constexpr bool AHEAD = NB < 4;
            auto v_at = [&](int s, int e) {
                const int key = kb + 8 * (s >> 2) + 4 * lk + (s & 3);
                return __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(vbuf, (key * kv_stride + NB * lq + e) * 4, 0, 0));
            };
            float ahead[AHEAD ? 16 : 1][NB];
            if constexpr (AHEAD) {
#pragma unroll
                for (int s = 0; s < 16; ++s)
#pragma unroll
                    for (int e = 0; e < NB; ++e) ahead[s][e] = v_at(s, e);
            }
            // lane half lk takes d = 8 t + 4 lk .. of each eight
            f32x16 s_acc = {};
#pragma unroll 4
            for (int t = 0; t < D / 8; ++t) {
                const int d = 8 * t + 4 * lk;
                const f32x4 kv = __builtin_bit_cast(
                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(kbuf, ((kb + lq) * kv_stride + d) * 4, 0, 0));
                const f32x4 qv = *(const f32x4*)(qrow + d);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s_acc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[i], qv[i] * p.qscale, s_acc, 0, 0, 0);
            }
            settle(s_acc);
            mask(s_acc, kb);
            const float corr = softmax(s_acc, 1.0f);
#pragma unroll
            for (int e = 0; e < NB; ++e)
#pragma unroll
                for (int r = 0; r < 16; ++r) o_acc[e][r] *= corr;
#pragma unroll
            for (int s = 0; s < 16; ++s)
#pragma unroll
                for (int e = 0; e < NB; ++e)
                    o_acc[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(AHEAD ? ahead[AHEAD ? s : 0][e] : v_at(s, e), s_acc[s],
                                                                    o_acc[e], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < NB; ++e) settle(o_acc[e]);
        }
    }

    if constexpr (KS > 1) {
        // waves of the odd blocks hand their O^T, m and l to those of the even
        // blocks (the loop's last barrier has retired every read of the keys)
        float* red = (float*)smem + wq * PER * 64 + lane;
        if (grp == 1) {
#pragma unroll
            for (int e = 0; e < NB; ++e)
#pragma unroll
                for (int r = 0; r < 16; ++r) red[(16 * e + r) * 64] = o_acc[e][r];
            red[16 * NB * 64] = m_run;
            red[(16 * NB + 1) * 64] = l_part;
        }
        __syncthreads();
        if (grp == 1) return;
        const float m1 = red[16 * NB * 64], l1 = red[(16 * NB + 1) * 64];
        const float m = fmaxf(m_run, m1);
        const float c0 = exp2_raw(m_run - m), c1 = exp2_raw(m1 - m);
        l_part = l_part * c0 + l1 * c1;
#pragma unroll
        for (int e = 0; e < NB; ++e)
#pragma unroll
            for (int r = 0; r < 16; ++r) o_acc[e][r] = o_acc[e][r] * c0 + red[(16 * e + r) * 64] * c1;
    }

    const float l_tot = l_part + __shfl_xor(l_part, 32);
    if (!q_valid) return;
    const float inv_l = 1.0f / l_tot;
    float* dst = Og + (size_t)q * row_stride + NB * 4 * lk;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int e = 0; e < NB; ++e) dst[NB * (8 * (r >> 2) + (r & 3)) + e] = o_acc[e][r] * inv_l;
}

template <int D, int KS>
int launch(lancius_hip_ctx* ctx, const AttnParams& p, unsigned tasks) {
    hipLaunchKernelGGL((attention_split<D, KS>), dim3(tasks), dim3(256 * KS), 0, ctx->stream, p);
    return check_launch(LANCIUS_KERNEL_NAME("attention_split D=%d x%d", D, KS));
}

}  // namespace

int launch_attention_split(lancius_hip_ctx* ctx, AttnParams& p) {
    p.q_tiles = (p.S + kQueries - 1) / kQueries;
    const size_t tasks = (size_t)p.q_tiles * p.H * p.Z;
    LANCIUS_REQUIRE(tasks < kMaxGridX, LANCIUS_HIP_ERR_SHAPE, "attention: too many tiles");
    const size_t cus = (size_t)cu_count(ctx);
    const bool ks2 = tasks <= cus;
    p.pair_tiles = p.causal && tasks <= 2 * cus;
    switch (p.D) {
        case 32: return ks2 ? launch<32, 2>(ctx, p, (unsigned)tasks) : launch<32, 1>(ctx, p, (unsigned)tasks);
        case 64: return ks2 ? launch<64, 2>(ctx, p, (unsigned)tasks) : launch<64, 1>(ctx, p, (unsigned)tasks);
        case 96: return ks2 ? launch<96, 2>(ctx, p, (unsigned)tasks) : launch<96, 1>(ctx, p, (unsigned)tasks);
        default: return ks2 ? launch<128, 2>(ctx, p, (unsigned)tasks) : launch<128, 1>(ctx, p, (unsigned)tasks);
    }
}

}  // namespace lancius
