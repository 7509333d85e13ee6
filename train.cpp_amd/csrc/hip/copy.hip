// Element-wise memory kernels: F32 fill (Device::fill_tensors) and the strided
// copy behind OP_DUP/OP_CPY/OP_CONT (compute_dup,
// src/backends/cpu/trc_cpu_ops.cpp:219-236). Both are HBM-bound streams; a copy
// is exact whatever order its elements move in.
#include "common.h"

namespace trc_hip {
namespace {

constexpr int CP_THREADS = 256;

__global__ __launch_bounds__(CP_THREADS) void k_fill_f32(float* __restrict__ dst, float value, int64_t n) {
    const int64_t stride = (int64_t) gridDim.x * CP_THREADS;
    for (int64_t i = (int64_t) blockIdx.x * CP_THREADS + threadIdx.x; i < n; i += stride) {
        dst[i] = value;
    }
}

// 16-byte stores for a 16-byte aligned dst; the last n % 4 floats go one by one.
__global__ __launch_bounds__(CP_THREADS) void k_fill_f32x4(f4* __restrict__ dst, float value, int64_t n4,
                                                          float* __restrict__ tail, int ntail) {
    const f4 v = {value, value, value, value};
    const int64_t stride = (int64_t) gridDim.x * CP_THREADS;
    for (int64_t i = (int64_t) blockIdx.x * CP_THREADS + threadIdx.x; i < n4; i += stride) dst[i] = v;
    if (blockIdx.x == 0 && (int) threadIdx.x < ntail) tail[threadIdx.x] = value;
}

// Copies element i of src to element i of dst in ggml linear order
// (tensor_offset_linear, src/core/trc_tensor.cpp:95-103), ne0 fastest, so a run of
// ne0 is one wave's contiguous read (or write) whenever that side has nb0 ==
// element size. Rows that run along ne0 on both sides in whole aligned 16-byte
// pieces are copied as such pieces. Bound by HBM, and by the launch up to about a
// megabyte; 64-bit divisions per 4-byte element took 30 us for the merge of 32 heads
// ([128, 512, 32, 4], 67 MB each way), 16-byte pieces and 32-bit multiplies 11 (6.2
// TB/s). One piece per lane: four took as long on large rows, 0.4 to 0.5 us more up
// to a megabyte ([64, 512] 2.30 -> 2.79), and up to twice as long where dst does not
// run along ne0 (1000 x 1001 written transposed 8.8 -> 16.9, [1000, 3, 500] 12.5 ->
// 26.3; only an order of four reversed dimensions gained, 64 each 243 -> 171).
template <typename T>
__global__ __launch_bounds__(CP_THREADS) void k_cpy32(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                     uint32_t total, FastDiv ne0, FastDiv ne1, FastDiv ne2,
                                                     int64_t snb0, int64_t snb1, int64_t snb2, int64_t snb3,
                                                     int64_t dnb0, int64_t dnb1, int64_t dnb2, int64_t dnb3) {
    const uint32_t idx = blockIdx.x * CP_THREADS + threadIdx.x;
    if (idx >= total) return;
    const uint32_t r = div_by(idx, ne0), i0 = idx - r * ne0.d;
    const uint32_t r2 = div_by(r, ne1), i1 = r - r2 * ne1.d;
    const uint32_t i3 = div_by(r2, ne2), i2 = r2 - i3 * ne2.d;
    *(T*) (dst + i0 * dnb0 + i1 * dnb1 + i2 * dnb2 + i3 * dnb3) =
        *(const T*) (src + i0 * snb0 + i1 * snb1 + i2 * snb2 + i3 * snb3);
}

// The same for 2^31 elements and more.
template <typename T>
__global__ __launch_bounds__(CP_THREADS) void k_cpy(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                   int64_t ne0, int64_t ne1, int64_t ne2, int64_t rows,
                                                   int64_t snb0, int64_t snb1, int64_t snb2, int64_t snb3,
                                                   int64_t dnb0, int64_t dnb1, int64_t dnb2, int64_t dnb3) {
    const int64_t total = ne0 * rows;
    const int64_t stride = (int64_t) gridDim.x * CP_THREADS;
    for (int64_t idx = (int64_t) blockIdx.x * CP_THREADS + threadIdx.x; idx < total; idx += stride) {
        const int64_t i0 = idx % ne0;
        const int64_t r = idx / ne0;
        const int64_t i1 = r % ne1;
        const int64_t i2 = (r / ne1) % ne2;
        const int64_t i3 = r / (ne1 * ne2);
        const T v = *(const T*) (src + i0 * snb0 + i1 * snb1 + i2 * snb2 + i3 * snb3);
        *(T*) (dst + i0 * dnb0 + i1 * dnb1 + i2 * dnb2 + i3 * dnb3) = v;
    }
}

// The same copy for 4-byte elements when src runs along dim 1 (nb1 == 4, the
// transposed views autograd builds) and dst along dim 0 (nb0 == 4): 64 x 64
// tiles of (i0, i1) go through LDS, read as 256-byte runs of src along i1 and
// written as 256-byte runs of dst along i0. Bound by the loads' latency where tiles
// are few: a thread asks for its 16 elements together, from addresses clamped into
// the tensor (each behind a branch of its own, they waited one for another:
// [64, 333, 12, 2] 4.7 -> 3.3 us again and again on one tensor, 6 us less of a pass
// whose product has just written it; 4095 x 4097 27.8 -> 23.9).
constexpr int TT = 64;
__global__ __launch_bounds__(CP_THREADS) void k_cpy_transpose(const uint8_t* __restrict__ src,
                                                             uint8_t* __restrict__ dst, int64_t ne0, int64_t ne1,
                                                             int64_t ne2, int64_t tiles0, int64_t tiles1,
                                                             int64_t snb0, int64_t snb2, int64_t snb3, int64_t dnb1,
                                                             int64_t dnb2, int64_t dnb3) {
    __shared__ uint32_t tile[TT][TT + 1];
    int64_t t = blockIdx.x;
    const int64_t t0 = t % tiles0;
    t /= tiles0;
    const int64_t t1 = t % tiles1;
    const int64_t plane = t / tiles1;
    const int64_t i2 = plane % ne2, i3 = plane / ne2;
    const uint8_t* sp = src + i2 * snb2 + i3 * snb3;
    uint8_t* dp = dst + i2 * dnb2 + i3 * dnb3;
    const int64_t b0 = t0 * TT, b1 = t1 * TT;
    const int lane = threadIdx.x % TT, row = threadIdx.x / TT;  // 4 rows per pass
    constexpr int STEP = CP_THREADS / TT;
    uint32_t v[TT / STEP];
    sp += (b1 + lane < ne1 ? b1 + lane : ne1 - 1) * 4;
#pragma unroll
    for (int k = 0; k < TT / STEP; ++k) {
        const int64_t i0 = b0 + row + k * STEP;
        v[k] = *(const uint32_t*) (sp + (i0 < ne0 ? i0 : ne0 - 1) * snb0);
    }
#pragma unroll
    for (int k = 0; k < TT / STEP; ++k) tile[row + k * STEP][lane] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TT; k += CP_THREADS / TT) {
        const int64_t i0 = b0 + lane, i1 = b1 + row + k;
        if (i0 < ne0 && i1 < ne1) *(uint32_t*) (dp + i0 * 4 + i1 * dnb1) = tile[lane][row + k];
    }
}

// k_cpy_transpose with 16-byte global accesses, for whole tiles (ne0 and ne1
// multiples of 64) of 16-byte aligned rows: a lane reads four floats along i1
// and writes four along i0; the tile is kept in LDS as [i1][i0].
constexpr int TL = TT + 4;  // LDS row stride in floats (keeps rows 16-byte aligned)
__global__ __launch_bounds__(CP_THREADS) void k_cpy_transpose4(const uint8_t* __restrict__ src,
                                                              uint8_t* __restrict__ dst, int64_t ne2,
                                                              int64_t tiles0, int64_t tiles1, int64_t snb0,
                                                              int64_t snb2, int64_t snb3, int64_t dnb1, int64_t dnb2,
                                                              int64_t dnb3) {
    __shared__ __attribute__((aligned(16))) float tile[TT * TL];
    int64_t t = blockIdx.x;
    const int64_t t0 = t % tiles0;
    t /= tiles0;
    const int64_t t1 = t % tiles1;
    const int64_t plane = t / tiles1;
    const int64_t i2 = plane % ne2, i3 = plane / ne2;
    const uint8_t* sp = src + i2 * snb2 + i3 * snb3 + t0 * TT * snb0 + t1 * TT * 4;
    uint8_t* dp = dst + i2 * dnb2 + i3 * dnb3 + t0 * TT * 4 + t1 * TT * dnb1;
    const int q = threadIdx.x % (TT / 4), row = threadIdx.x / (TT / 4);  // 16 rows per pass
#pragma unroll
    for (int k = 0; k < TT; k += CP_THREADS / (TT / 4)) {
        const f4 v = *(const f4*) (sp + (row + k) * snb0 + q * 16);  // src row i0 = row + k, i1 = 4q .. 4q + 3
#pragma unroll
        for (int c = 0; c < 4; ++c) tile[(4 * q + c) * TL + row + k] = v[c];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TT; k += CP_THREADS / (TT / 4)) {
        // dst row i1 = row + k, i0 = 4q .. 4q + 3
        *(f4*) (dp + (row + k) * dnb1 + q * 16) = *(const f4*) (tile + (row + k) * TL + 4 * q);
    }
}

unsigned grid_for(int64_t n) {
    const int64_t want = (n + CP_THREADS - 1) / CP_THREADS;
    return (unsigned) (want < 65536 ? (want > 0 ? want : 1) : 65536);
}

}  // namespace

int launch_fill_f32(float* dst, float value, int64_t count, hipStream_t stream) {
    if ((((uintptr_t) dst) & 15u) == 0) {
        const int64_t n4 = count / 4;
        hipLaunchKernelGGL(k_fill_f32x4, dim3(grid_for(n4)), dim3(CP_THREADS), 0, stream, (f4*) dst, value, n4,
                           dst + 4 * n4, (int) (count - 4 * n4));
    } else {
        hipLaunchKernelGGL(k_fill_f32, dim3(grid_for(count)), dim3(CP_THREADS), 0, stream, dst, value, count);
    }
    return check_launch("fill_f32");
}

int launch_cpy(const trc_hip_tensor& s, const trc_hip_tensor& d, size_t es, hipStream_t stream) {
    const int64_t rows = s.ne[1] * s.ne[2] * s.ne[3];
    const int64_t n = s.ne[0] * rows;
    const uint8_t* sp = (const uint8_t*) s.data;
    uint8_t* dp = (uint8_t*) d.data;
    // (up to 12 runs of src fill too little of a tile: 3 of 100000 6.1 us, by element 2.6,
    // 12 of 2000000 65 and 52; 16 of 2000000 67 and 82)
    if (es == 4 && s.nb[1] == 4 && d.nb[0] == 4 && s.ne[0] > 12 && s.ne[1] > 1) {
        const int64_t tiles0 = (s.ne[0] + TT - 1) / TT, tiles1 = (s.ne[1] + TT - 1) / TT;
        const int64_t grid = tiles0 * tiles1 * s.ne[2] * s.ne[3];
        const bool whole = s.ne[0] % TT == 0 && s.ne[1] % TT == 0 && (((uintptr_t) sp | (uintptr_t) dp) & 15u) == 0 &&
                           s.nb[0] % 16 == 0 && d.nb[1] % 16 == 0 && s.nb[2] % 16 == 0 && s.nb[3] % 16 == 0 &&
                           d.nb[2] % 16 == 0 && d.nb[3] % 16 == 0;
        if (grid <= max_groups(CP_THREADS) && whole) {
            hipLaunchKernelGGL(k_cpy_transpose4, dim3((unsigned) grid), dim3(CP_THREADS), 0, stream, sp, dp, s.ne[2],
                               tiles0, tiles1, (int64_t) s.nb[0], (int64_t) s.nb[2], (int64_t) s.nb[3],
                               (int64_t) d.nb[1], (int64_t) d.nb[2], (int64_t) d.nb[3]);
            return check_launch("cpy (transpose)");
        }
        if (grid <= max_groups(CP_THREADS)) {
            hipLaunchKernelGGL(k_cpy_transpose, dim3((unsigned) grid), dim3(CP_THREADS), 0, stream, sp, dp, s.ne[0],
                               s.ne[1], s.ne[2], tiles0, tiles1, (int64_t) s.nb[0], (int64_t) s.nb[2],
                               (int64_t) s.nb[3], (int64_t) d.nb[1], (int64_t) d.nb[2], (int64_t) d.nb[3]);
            return check_launch("cpy (transpose)");
        }
    }
    if (n < ((int64_t) 1 << 31) - CP_THREADS) {
        // whole 16-byte pieces of rows that run along ne0 on both sides
        uintptr_t bits = (uintptr_t) sp | (uintptr_t) dp | (uintptr_t) (s.ne[0] * (int64_t) es);
        for (int k = 1; k < 4; ++k) {
            if (s.ne[k] > 1) bits |= (uintptr_t) s.nb[k] | (uintptr_t) d.nb[k];
        }
        const bool run = s.ne[0] == 1 || (s.nb[0] == es && d.nb[0] == es);
        const size_t w = run && (bits & 15u) == 0 ? 16 : es;
        const int64_t ne0 = s.ne[0] * (int64_t) es / (int64_t) w;
        const int64_t snb0 = w == 16 ? 16 : (int64_t) s.nb[0], dnb0 = w == 16 ? 16 : (int64_t) d.nb[0];
        const uint32_t total = (uint32_t) (ne0 * rows);
        const dim3 grid((total + CP_THREADS - 1) / CP_THREADS);
#define TRC_CPY32(T)                                                                                             \
    hipLaunchKernelGGL(k_cpy32<T>, grid, dim3(CP_THREADS), 0, stream, sp, dp, total, fast_div(ne0),              \
                       fast_div(s.ne[1]), fast_div(s.ne[2]), snb0, (int64_t) s.nb[1], (int64_t) s.nb[2],         \
                       (int64_t) s.nb[3], dnb0, (int64_t) d.nb[1], (int64_t) d.nb[2], (int64_t) d.nb[3])
        switch (w) {
            case 1: TRC_CPY32(uint8_t); break;
            case 2: TRC_CPY32(uint16_t); break;
            case 4: TRC_CPY32(uint32_t); break;
            case 8: TRC_CPY32(uint64_t); break;
            default: TRC_CPY32(f4); break;
        }
#undef TRC_CPY32
        return check_launch("cpy");
    }
#define TRC_CPY_ARGS                                                                                        \
    dim3(grid_for(n)), dim3(CP_THREADS), 0, stream, sp, dp, s.ne[0], s.ne[1], s.ne[2], rows,                \
        (int64_t) s.nb[0], (int64_t) s.nb[1], (int64_t) s.nb[2], (int64_t) s.nb[3], (int64_t) d.nb[0],      \
        (int64_t) d.nb[1], (int64_t) d.nb[2], (int64_t) d.nb[3]
    switch (es) {
        case 1: hipLaunchKernelGGL(k_cpy<uint8_t>, TRC_CPY_ARGS); break;
        case 2: hipLaunchKernelGGL(k_cpy<uint16_t>, TRC_CPY_ARGS); break;
        case 4: hipLaunchKernelGGL(k_cpy<uint32_t>, TRC_CPY_ARGS); break;
        default: hipLaunchKernelGGL(k_cpy<uint64_t>, TRC_CPY_ARGS); break;
    }
#undef TRC_CPY_ARGS
    return check_launch("cpy");
}

}  // namespace trc_hip
