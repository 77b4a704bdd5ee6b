// Reductions and the 2-D transpose of the scheduler dispatch
// (bleeding/v11A1/src/runtime/lancius_scheduler.c:246-267): TRANSPOSE, SUM,
// SUM_AXIS0, SUM_AXIS1.  All HBM-bound.
//
// Sums accumulate in fp64 (the reference's accumulator type) and store fp32.
// Every element goes to a partial chosen from the shape alone and partials
// are combined in a fixed order, so results are bit-identical from run to
// run; no atomics.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace lancius {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ double block_sum(double v, double* part) {
    part[threadIdx.x] = v;
    __syncthreads();
    for (int w = kThreads / 2; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    return part[0];
}

// SUM, first stage: workgroup b sums the float4 groups b*256+t, then every
// gridDim*256-th after it (fixed by n and the grid), plus the n % 4 tail in
// workgroup 0.
__global__ void __launch_bounds__(kThreads) sum_partials(double* __restrict__ partial, const float* __restrict__ in,
                                                         size_t n, int vec) {
    __shared__ double part[kThreads];
    const size_t stride = (size_t)gridDim.x * kThreads;
    double t = 0.0;
    if (vec) {
        const size_t n4 = n / 4;
        for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n4; i += stride) {
            const f32x4 v = ((const f32x4*)in)[i];
            t += ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
        }
        if (blockIdx.x == 0 && threadIdx.x < n - 4 * n4) t += (double)in[4 * n4 + threadIdx.x];
    } else {
        for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += stride) t += (double)in[i];
    }
    const double s = block_sum(t, part);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(kThreads) sum_finish(float* __restrict__ out, const double* __restrict__ partial,
                                                       int count) {
    __shared__ double part[kThreads];
    double t = 0.0;
    for (int i = threadIdx.x; i < count; i += kThreads) t += partial[i];
    const double s = block_sum(t, part);
    if (threadIdx.x == 0) out[0] = (float)s;
}

// SUM_AXIS0 over rows [r0, r1) of split blockIdx.y (T: the values, or the
// splits' partial sums).  A workgroup takes w columns (16, 32 or 64: rows of
// few columns still fill its waves); its 512 / w row groups each add every
// (512 / w)-th row, eight loads in flight, and are then added in a fixed
// order, in the wave by shuffles and over the eight waves through LDS.
// Bound by the loads' latency: one column per thread over all rows of a split
// was a chain of 64 to 512 dependent adds behind single loads (64 x 128:
// 7.3 us a call, now 3.9; 512 x 128 49 us, now 5.8; 2048 x 4096 29, now 9.5).
constexpr int kAxis0Threads = 512;
constexpr int kAxis0Unroll = 8;
template <typename T>
__global__ void __launch_bounds__(kAxis0Threads) sum_axis0(float* __restrict__ out, double* __restrict__ partial,
                                                           const T* __restrict__ in, size_t rows, size_t cols,
                                                           size_t rchunk, int w) {
    __shared__ double part[kAxis0Threads];
    const size_t groups = kAxis0Threads / w;
    const size_t r0 = (size_t)blockIdx.y * rchunk;
    const size_t r1 = std::min(rows, r0 + rchunk);
    for (size_t c0 = (size_t)blockIdx.x * w; c0 < cols; c0 += (size_t)gridDim.x * w) {
        const size_t c = c0 + (threadIdx.x & (w - 1));
        const T* __restrict__ x = in + std::min(c, cols - 1);
        double t = 0.0;
        for (size_t r = r0 + threadIdx.x / w; r < r1; r += kAxis0Unroll * groups) {
            T v[kAxis0Unroll];
#pragma unroll
            for (int i = 0; i < kAxis0Unroll; ++i) v[i] = x[std::min(r + i * groups, r1 - 1) * cols];
#pragma unroll
            for (int i = 0; i < kAxis0Unroll; ++i) t += r + i * groups < r1 ? (double)v[i] : 0.0;
        }
        for (int off = w; off < 64; off <<= 1) t += __shfl_xor(t, off);
        part[threadIdx.x] = t;
        __syncthreads();
        if ((int)threadIdx.x < w && c < cols) {
            t = 0.0;
#pragma unroll
            for (int i = 0; i < kAxis0Threads; i += 64) t += part[threadIdx.x + i];
            if (gridDim.y == 1)
                out[c] = (float)t;
            else
                partial[(size_t)blockIdx.y * cols + c] = t;
        }
        __syncthreads();
    }
}

// SUM_AXIS0 of a few rows: a column per thread.
__global__ void __launch_bounds__(kThreads) sum_axis0_columns(float* __restrict__ out, const float* __restrict__ in,
                                                              int rows, size_t cols) {
    const size_t c = (size_t)blockIdx.x * kThreads + threadIdx.x;
    if (c >= cols) return;
    double t = 0.0;
    for (int r = 0; r < rows; ++r) t += (double)in[(size_t)r * cols + c];
    out[c] = (float)t;
}

// SUM_AXIS1: one wave per row, lanes strided over the columns, fp64 wave sum.
__global__ void __launch_bounds__(kThreads) sum_axis1_rows(float* __restrict__ out, const float* __restrict__ in,
                                                           size_t rows, size_t cols) {
    const size_t row = (size_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float* x = in + row * cols;
    double t = 0.0;
    for (size_t c = lane; c < cols; c += 64) t += (double)x[c];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) t += __shfl_xor(t, off);
    if (lane == 0) out[row] = (float)t;
}

// TRANSPOSE through a 64x65 LDS tile: reads and writes are both 64-float
// row segments.  Tiles are numbered along columns of the input first.
__global__ void __launch_bounds__(kThreads) transpose_tiles(float* __restrict__ out, const float* __restrict__ in,
                                                            size_t rows, size_t cols, size_t tiles_c) {
    __shared__ float t[64][65];
    const size_t tile = blockIdx.x;
    const size_t r0 = (tile / tiles_c) * 64, c0 = (tile % tiles_c) * 64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const size_t r = r0 + ty + 4 * i, c = c0 + tx;
        if (r < rows && c < cols) t[ty + 4 * i][tx] = in[r * cols + c];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const size_t c = c0 + ty + 4 * i, r = r0 + tx;  // out row c, column r
        if (r < rows && c < cols) out[c * rows + r] = t[tx][ty + 4 * i];
    }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace
}  // namespace lancius

using namespace lancius;

extern "C" {

int lancius_hip_sum_f32(lancius_hip_ctx* ctx, float* out, const float* in, size_t n) {
    LANCIUS_REQUIRE(ctx && out && in, LANCIUS_HIP_ERR_NULL_PTR, "sum: NULL argument");
    if (int rc = bind_device(ctx)) return rc;
    // Enough workgroups to stream from every CU, each with >= 4096 values.
    const size_t blocks = std::max<size_t>(1, std::min<size_t>(1024, (n + 4095) / 4096));
    void* ws = nullptr;
    if (int rc = workspace(ctx, blocks * sizeof(double), &ws)) return rc;
    hipLaunchKernelGGL(sum_partials, dim3((unsigned)blocks), dim3(kThreads), 0, ctx->stream, (double*)ws, in, n,
                       (int)aligned16(in));
    if (int rc = check_launch("sum_partials")) return rc;
    hipLaunchKernelGGL(sum_finish, dim3(1), dim3(kThreads), 0, ctx->stream, out, (const double*)ws, (int)blocks);
    return check_launch("sum_finish");
}

int lancius_hip_sum_axis0_f32(lancius_hip_ctx* ctx, float* out, const float* in, size_t rows, size_t cols) {
    LANCIUS_REQUIRE(ctx && out && in, LANCIUS_HIP_ERR_NULL_PTR, "sum_axis0: NULL argument");
    if (cols == 0) return ok();
    if (int rc = bind_device(ctx)) return rc;
    LANCIUS_REQUIRE((cols + kThreads - 1) / kThreads < kMaxGridX, LANCIUS_HIP_ERR_SHAPE, "sum_axis0: %zu columns", cols);
    // Few rows with columns enough for one each per thread: no partial sums
    // to add (16 x 2^20: 13.6 us, 40 with sum_axis0; 33 x 2^17: 5.0, 6.8; 64 x 2^18:
    // 20.3, 11.5).
    if (rows <= 48 && cols >= (1u << 16)) {
        hipLaunchKernelGGL(sum_axis0_columns, dim3((unsigned)((cols + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                           ctx->stream, out, in, (int)rows, cols);
        return check_launch("sum_axis0_columns");
    }
    const int w = cols <= 16 ? 16 : cols <= 32 ? 32 : 64;
    const size_t col_blocks = (cols + w - 1) / w, groups = kAxis0Threads / w;
    // Row splits: ~1024 workgroups in all, each thread over >= 16 rows; none
    // while a thread has up to 64, where a second launch would cost more than
    // it saves (512 x 128: 5.8 us in one, 513 x 128 6.5 in two).
    size_t splits = rows <= 64 * groups ? 1 : std::max<size_t>(1, std::min<size_t>(rows / (16 * groups), 1024 / col_blocks));
    splits = std::min<size_t>(splits, 65535);
    const size_t rchunk = rows ? (rows + splits - 1) / splits : 1;
    splits = rows ? (rows + rchunk - 1) / rchunk : 1;
    const unsigned grid_x = (unsigned)std::min<size_t>(col_blocks, 1u << 22);  // 2^31 work-items
    double* ws = nullptr;
    if (splits > 1)
        if (int rc = workspace(ctx, splits * cols * sizeof(double), (void**)&ws)) return rc;
    hipLaunchKernelGGL(sum_axis0<float>, dim3(grid_x, (unsigned)splits), dim3(kAxis0Threads), 0,
                       ctx->stream, out, ws, in, rows, cols, rchunk, w);
    if (int rc = check_launch("sum_axis0")) return rc;
    if (splits > 1) {
        hipLaunchKernelGGL(sum_axis0<double>, dim3(grid_x), dim3(kAxis0Threads), 0, ctx->stream, out,
                           nullptr, (const double*)ws, splits, cols, splits, w);
        if (int rc = check_launch("sum_axis0")) return rc;
    }
    return ok();
}

int lancius_hip_sum_axis1_f32(lancius_hip_ctx* ctx, float* out, const float* in, size_t rows, size_t cols) {
    LANCIUS_REQUIRE(ctx && out && in, LANCIUS_HIP_ERR_NULL_PTR, "sum_axis1: NULL argument");
    if (rows == 0) return ok();
    if (int rc = bind_device(ctx)) return rc;
    const size_t blocks = (rows + 3) / 4;
    LANCIUS_REQUIRE(blocks < kMaxGridX, LANCIUS_HIP_ERR_SHAPE, "sum_axis1: %zu rows", rows);
    hipLaunchKernelGGL(sum_axis1_rows, dim3((unsigned)blocks), dim3(kThreads), 0, ctx->stream, out, in, rows, cols);
    return check_launch("sum_axis1");
}

int lancius_hip_transpose_f32(lancius_hip_ctx* ctx, float* out, const float* in, size_t rows, size_t cols) {
    LANCIUS_REQUIRE(ctx && out && in, LANCIUS_HIP_ERR_NULL_PTR, "transpose: NULL argument");
    if (rows == 0 || cols == 0) return ok();
    if (int rc = bind_device(ctx)) return rc;
    const size_t tr = (rows + 63) / 64, tc = (cols + 63) / 64;
    LANCIUS_REQUIRE(tr * tc < kMaxGridX, LANCIUS_HIP_ERR_SHAPE, "transpose: %zu x %zu", rows, cols);
    hipLaunchKernelGGL(transpose_tiles, dim3((unsigned)(tr * tc)), dim3(kThreads), 0, ctx->stream, out, in, rows, cols,
                       tc);
    return check_launch("transpose");
}

}  // extern "C"
