// F32 element-wise graph ops that a Linear layer's forward and autograd
// backward put around mul_mat on the device: ADD and MUL with ggml broadcast,
// ACC into a strided region, REPEAT_BACK, REPEAT, and SUM (the scalar loss).
// Each output element is produced by the same single float operation, or the
// same ordered sum, as the reference CPU kernels, so the results are
// bit-identical:
//   add, mul     src/ops/trc_ops.cpp:19-32,46,59; compute_binary
//                src/backends/cpu/trc_cpu_ops.cpp:52-78 (offset_broadcast :18-28)
//   acc          src/core/trc_tensor.cpp:322-361; compute_acc trc_cpu_ops.cpp:954-999
//   repeat_back  src/ops/trc_ops.cpp:458-470; compute_repeat_back trc_cpu_ops.cpp:932-952
//   repeat       src/ops/trc_ops.cpp:447-456; compute_repeat trc_cpu_ops.cpp:913-928
//   sum          src/ops/trc_ops.cpp:214-221; compute_sum trc_cpu_ops.cpp:302-315
//                (row_sum_f32 :284-300)
//
// Mapping: one workgroup row-loop per ggml row (ne0-run); lanes stride over the
// row, so loads and stores along ne0 are coalesced whenever nb0 == 4.
#include "common.h"

namespace trc_hip {
namespace {

constexpr int EW_THREADS = 256;

struct Shape4 {
    int64_t ne[4];
    int64_t nb[4];  // bytes
};

Shape4 shape_of(const trc_hip_tensor& t) {
    Shape4 s;
    for (int d = 0; d < 4; ++d) {
        s.ne[d] = t.ne[d];
        s.nb[d] = (int64_t) t.nb[d];
    }
    return s;
}

enum class BinOp { ADD, MUL };

// dst[i] = a[i] (+ or *) b[broadcast(i)], rows of dst distributed over the grid
template <BinOp OP>
__global__ __launch_bounds__(EW_THREADS) void k_binary(const uint8_t* __restrict__ a, Shape4 sa,
                                                       const uint8_t* __restrict__ b, Shape4 sb,
                                                       uint8_t* __restrict__ d, Shape4 sd) {
    const int64_t rows = sd.ne[1] * sd.ne[2] * sd.ne[3];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sd.ne[1], i2 = (r / sd.ne[1]) % sd.ne[2], i3 = r / (sd.ne[1] * sd.ne[2]);
        const uint8_t* pa = a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3];
        const uint8_t* pb = b + (sb.ne[1] == 1 ? 0 : i1 * sb.nb[1]) + (sb.ne[2] == 1 ? 0 : i2 * sb.nb[2]) +
                            (sb.ne[3] == 1 ? 0 : i3 * sb.nb[3]);
        uint8_t* pd = d + i1 * sd.nb[1] + i2 * sd.nb[2] + i3 * sd.nb[3];
        const int64_t bnb0 = sb.ne[0] == 1 ? 0 : sb.nb[0];
        for (int64_t i0 = threadIdx.x; i0 < sd.ne[0]; i0 += EW_THREADS) {
            const float va = *(const float*) (pa + i0 * sa.nb[0]), vb = *(const float*) (pb + i0 * bnb0);
            *(float*) (pd + i0 * sd.nb[0]) = OP == BinOp::ADD ? va + vb : va * vb;
        }
    }
}

// k_binary with four floats per lane: rows of a, d (and b, unless b broadcasts
// along ne0) are 16-byte aligned with nb0 == 4 and ne0 % 4 == 0. The same single
// rounding per element.
template <BinOp OP>
__global__ __launch_bounds__(EW_THREADS) void k_binary4(const uint8_t* __restrict__ a, Shape4 sa,
                                                        const uint8_t* __restrict__ b, Shape4 sb,
                                                        uint8_t* __restrict__ d, Shape4 sd) {
    const int64_t rows = sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int64_t n4 = sd.ne[0] / 4;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sd.ne[1], i2 = (r / sd.ne[1]) % sd.ne[2], i3 = r / (sd.ne[1] * sd.ne[2]);
        const f4* pa = (const f4*) (a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3]);
        const uint8_t* pb = b + (sb.ne[1] == 1 ? 0 : i1 * sb.nb[1]) + (sb.ne[2] == 1 ? 0 : i2 * sb.nb[2]) +
                            (sb.ne[3] == 1 ? 0 : i3 * sb.nb[3]);
        f4* pd = (f4*) (d + i1 * sd.nb[1] + i2 * sd.nb[2] + i3 * sd.nb[3]);
        for (int64_t q = threadIdx.x; q < n4; q += EW_THREADS) {
            const f4 va = pa[q];
            f4 vb;
            if (sb.ne[0] == 1) {
                const float x = *(const float*) pb;
                vb = (f4){x, x, x, x};
            } else {
                vb = ((const f4*) pb)[q];
            }
            pd[q] = OP == BinOp::ADD ? va + vb : va * vb;
        }
    }
}

enum class UnOp { SQR, SCALE };

// dst[i] = a[i] * a[i] (SQR: fn_sqr, src/backends/cpu/trc_cpu_ops.cpp:86, through
// compute_unary :119-135) or a[i] * s (SCALE: compute_scale :140-150), element i
// of dst from element i of a (same shape, any strides): one float multiply each,
// rows of dst distributed over the grid as in k_binary
template <UnOp OP>
__global__ __launch_bounds__(EW_THREADS) void k_unary(const uint8_t* __restrict__ a, Shape4 sa,
                                                      uint8_t* __restrict__ d, Shape4 sd, float s) {
    const int64_t rows = sd.ne[1] * sd.ne[2] * sd.ne[3];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sd.ne[1], i2 = (r / sd.ne[1]) % sd.ne[2], i3 = r / (sd.ne[1] * sd.ne[2]);
        const uint8_t* pa = a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3];
        uint8_t* pd = d + i1 * sd.nb[1] + i2 * sd.nb[2] + i3 * sd.nb[3];
        for (int64_t i0 = threadIdx.x; i0 < sd.ne[0]; i0 += EW_THREADS) {
            const float v = *(const float*) (pa + i0 * sa.nb[0]);
            *(float*) (pd + i0 * sd.nb[0]) = OP == UnOp::SQR ? v * v : v * s;
        }
    }
}

// k_unary with four floats per lane (rows of a and d 16-byte aligned, nb0 == 4,
// ne0 % 4 == 0); the same single rounding per element
template <UnOp OP>
__global__ __launch_bounds__(EW_THREADS) void k_unary4(const uint8_t* __restrict__ a, Shape4 sa,
                                                       uint8_t* __restrict__ d, Shape4 sd, float s) {
    const int64_t rows = sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int64_t n4 = sd.ne[0] / 4;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sd.ne[1], i2 = (r / sd.ne[1]) % sd.ne[2], i3 = r / (sd.ne[1] * sd.ne[2]);
        const f4* pa = (const f4*) (a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3]);
        f4* pd = (f4*) (d + i1 * sd.nb[1] + i2 * sd.nb[2] + i3 * sd.nb[3]);
        for (int64_t q = threadIdx.x; q < n4; q += EW_THREADS) {
            const f4 v = pa[q];
            pd[q] = OP == UnOp::SQR ? v * v : v * s;
        }
    }
}

// The same operations where every operand is one contiguous run of n floats (16-byte
// aligned): float4s with no rows to find, which rows of odd lengths leave to single
// floats otherwise, and every lane busy whatever ne0 is. NT: the result is larger
// than the caches and is stored past them (268 MB scaled: 102 -> 85 us).
enum class FlatOp { ADD, MUL, SQR, SCALE };
constexpr int64_t FLAT_NT = (int64_t) 32 << 20;  // floats
template <FlatOp OP, bool NT>
__global__ __launch_bounds__(EW_THREADS) void k_flat(const f4* a, const f4* b, f4* d, int64_t n, float s) {
    auto one = [&](auto x, auto y) {
        if constexpr (OP == FlatOp::ADD) return x + y;
        else if constexpr (OP == FlatOp::MUL) return x * y;
        else if constexpr (OP == FlatOp::SQR) return x * x;
        else return x * s;
    };
    constexpr bool TWO = OP == FlatOp::ADD || OP == FlatOp::MUL;
    const int64_t q = (int64_t) blockIdx.x * EW_THREADS + threadIdx.x;
    if (q < n / 4) {
        const f4 va = a[q], v = one(va, TWO ? b[q] : va);
        if constexpr (NT) __builtin_nontemporal_store(v, d + q);
        else d[q] = v;
    } else if (q == n / 4) {  // the last n % 4
        for (int64_t i = n / 4 * 4; i < n; ++i) {
            const float x = ((const float*) a)[i];
            ((float*) d)[i] = one(x, TWO ? ((const float*) b)[i] : x);
        }
    }
}

// k_repeat for a dst whose rows are 16-byte aligned with nb0 == 4 and ne0 % 4 ==
// 0: one row of dst per workgroup pass, four floats per lane and store.
__global__ __launch_bounds__(EW_THREADS) void k_repeat4(const uint8_t* __restrict__ a, Shape4 sa,
                                                        uint8_t* __restrict__ d, Shape4 sd) {
    const int64_t rows = sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int64_t n4 = sd.ne[0] / 4;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sd.ne[1], i2 = (r / sd.ne[1]) % sd.ne[2], i3 = r / (sd.ne[1] * sd.ne[2]);
        const uint8_t* pa = a + (i1 % sa.ne[1]) * sa.nb[1] + (i2 % sa.ne[2]) * sa.nb[2] + (i3 % sa.ne[3]) * sa.nb[3];
        f4* pd = (f4*) (d + i1 * sd.nb[1] + i2 * sd.nb[2] + i3 * sd.nb[3]);
        if (sa.ne[0] == 1) {  // one value per row of dst (e.g. a loss gradient spread out)
            const float x = *(const float*) pa;
            for (int64_t q = threadIdx.x; q < n4; q += EW_THREADS) pd[q] = (f4){x, x, x, x};
            continue;
        }
        for (int64_t q = threadIdx.x; q < n4; q += EW_THREADS) {
            f4 v;
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = *(const float*) (pa + ((4 * q + c) % sa.ne[0]) * sa.nb[0]);
            pd[q] = v;
        }
    }
}

// dst[i] = a[i mod a.ne, per dim]: every dim of a is 1 (broadcast) or dst's
// extent; one thread per dst element, grid-stride
__global__ __launch_bounds__(EW_THREADS) void k_repeat(const uint8_t* __restrict__ a, Shape4 sa,
                                                       uint8_t* __restrict__ d, Shape4 sd) {
    const int64_t n = sd.ne[0] * sd.ne[1] * sd.ne[2] * sd.ne[3];
    for (int64_t j = (int64_t) blockIdx.x * EW_THREADS + threadIdx.x; j < n; j += (int64_t) gridDim.x * EW_THREADS) {
        int64_t rem = j, oa = 0, od = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int64_t idx = rem % sd.ne[k];
            rem /= sd.ne[k];
            oa += (sa.ne[k] == 1 ? 0 : idx % sa.ne[k]) * sa.nb[k];
            od += idx * sd.nb[k];
        }
        *(float*) (d + od) = *(const float*) (a + oa);
    }
}

// *d = sum of a, as compute_sum forms it: each row (ne0-run) summed from 0 in
// double in element order, the row sums added in double in row order (i1
// fastest, then i2, i3), one rounding to float at the end.
//
// Rows of 64 elements and more (k_sum_rows_lds) stream through LDS and meet in the
// workgroup that finishes last, unless the sum in any order settles the result
// (k_sum_bounded below). Shorter rows take two launches: k_sum_rows, one
// lane per row with the row's next SR_AHEAD loads issued ahead of the adds (from
// addresses clamped into the row, so no branch waits on them), then k_sum_combine,
// one wave that adds the row sums in row order. k_sum (one workgroup, no
// workspace) serves the row counts the workspace cannot hold.
constexpr int SR_THREADS = 64;
constexpr int SR_AHEAD = 32;

template <bool VEC>
__global__ __launch_bounds__(SR_THREADS) void k_sum_rows(const uint8_t* __restrict__ a, Shape4 sa,
                                                         double* __restrict__ part) {
    const int64_t rows = sa.ne[1] * sa.ne[2] * sa.ne[3];
    const int64_t r = (int64_t) blockIdx.x * SR_THREADS + threadIdx.x;
    if (r >= rows) return;  // no barrier below
    const int64_t i1 = r % sa.ne[1], i2 = (r / sa.ne[1]) % sa.ne[2], i3 = r / (sa.ne[1] * sa.ne[2]);
    const uint8_t* p = a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3];
    const int64_t n = sa.ne[0];
    double s = 0.0;
    if constexpr (VEC) {  // nb0 == 4, every row 16-byte aligned
        const f4* q = (const f4*) p;
        const int64_t n4 = n / 4;
        if (n4 > 0) {
            f4 buf[SR_AHEAD];
#pragma unroll
            for (int u = 0; u < SR_AHEAD; ++u) buf[u] = q[u < n4 ? u : n4 - 1];
            for (int64_t i = 0; i < n4; i += SR_AHEAD) {
#pragma unroll
                for (int u = 0; u < SR_AHEAD; ++u) {
                    if (i + u < n4) {  // the same for every lane: rows have one length
                        const f4 v = buf[u];
                        s = s + (double) v.x;
                        s = s + (double) v.y;
                        s = s + (double) v.z;
                        s = s + (double) v.w;
                    }
                    const int64_t nx = i + SR_AHEAD + u;
                    buf[u] = q[nx < n4 ? nx : n4 - 1];
                }
            }
        }
        for (int64_t i0 = 4 * n4; i0 < n; ++i0) s = s + (double) ((const float*) p)[i0];
    } else {
        float buf[SR_AHEAD];
#pragma unroll
        for (int u = 0; u < SR_AHEAD; ++u) buf[u] = *(const float*) (p + (u < n ? u : n - 1) * sa.nb[0]);
        for (int64_t i = 0; i < n; i += SR_AHEAD) {
#pragma unroll
            for (int u = 0; u < SR_AHEAD; ++u) {
                if (i + u < n) s = s + (double) buf[u];
                const int64_t nx = i + SR_AHEAD + u;
                buf[u] = *(const float*) (p + (nx < n ? nx : n - 1) * sa.nb[0]);
            }
        }
    }
    part[r] = s;
}

// Row sums with the loads spread over a whole workgroup: SB_ROWS rows per
// workgroup stream through an LDS ring of SB_D chunks of SB_C elements per row,
// loaded by all SB_THREADS threads (float4s where VEC: nb0 == 4, whole float4s, rows
// 16-byte aligned; else element by element, still in runs along the row) SB_D - 1
// chunks ahead of the lanes that hold the rows' sums; lane r of wave 0 adds row r's
// chunk in element order. With SB_D >= 3 one barrier per chunk separates a slot's
// reads from its next fill. The threads that stage a chunk convert it to double
// (exact) as they store it, so the lanes on the chain issue only the adds, and
// store zeros past the row's end, which change no sum (it is never -0: it starts
// from +0). What remains is the chain itself: each dependent v_add_f64 waits ~15
// cycles for the one before. 130 rows of 777 unaligned floats: 50 us with one lane
// per row, 13 here.
// The workgroup that takes the last ticket adds the row sums in row order (512
// rows of 4096 40.0 us with a launch of its own for that, 37.2 here).
// CHECKED: runs behind k_sum_bounded, whose sums may make all of this unnecessary.
constexpr int SB_ROWS = 8;
constexpr int SB_THREADS = 256;
constexpr int SB_C = 256;
constexpr int SB_LD = SB_C + 2;  // padded row (in doubles) of an LDS slot: rows 4 banks apart
constexpr int SB_MIN = 64;       // shorter rows: one lane each
typedef double sb_d2 __attribute__((ext_vector_type(2)));
constexpr int SB_D = 4;
constexpr int SB_RING = SB_D * SB_ROWS * SB_LD;

// s + the first n doubles (n a multiple of 16) at p, in order: the next 16 are read
// from LDS while the current 16 are added
__device__ __forceinline__ double sum_chain(double s, const double* p, int n) {
    const sb_d2* q = (const sb_d2*) p;
    sb_d2 cur[8], nxt[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) cur[k] = q[k];
    for (int g = 16; g < n; g += 16) {
#pragma unroll
        for (int k = 0; k < 8; ++k) nxt[k] = q[g / 2 + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            s = s + cur[k].x;
            s = s + cur[k].y;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) cur[k] = nxt[k];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        s = s + cur[k].x;
        s = s + cur[k].y;
    }
    return s;
}

// The chain above is what the order of the sum costs, and mostly the order does not
// matter: one pass over contiguous data gives S, its sum in double in some order, and
// A, the sum of the magnitudes. With u = 2^-53 and at most k roundings on an
// element's way into either sum, both lie within k u A (1 + k u) of the true sum (N.
// J. Higham, "Accuracy and Stability of Numerical Algorithms", 4.2), so the sum in
// the stated order lies within b of S, b = 1.01 u A times the k of both orders and a
// few for the check's own roundings. Rounding to float is monotone: where S - b and
// S + b round to the same float, so does the sum in order, and that float is its
// result bit for bit. Elsewhere (A not finite, or S within b of the middle of two
// floats: about k u A / (6e-8 |S|) of all sums, 2e-5 of the sums of 512 x 4096
// squares) the chain runs as without this.
// S and A stay one pair per workgroup; every workgroup of the second launch adds
// the pairs up in one order and comes to the same decision, so that no ticket, flag
// or wait lies between. Bound by two launches, then by HBM (65536 x 4096 5.6 TB/s).
// Chain -> here, both launches: [777, 130] 13.0 -> 6.7 us, [4096, 512] 37.2 -> 6.8,
// [333, 7992 rows] 68.5 -> 7.5, [4096, 65536] 954 -> 191; where the chain has to run
// all the same, 4.5 us more, and a fifth more for long 16-byte aligned rows of which there
// are few (its loop is not unrolled: one row of 100000 555 -> 680; unrolled, 590, but
// [4096, 4096] with its many workgroups 75 -> 94).
constexpr int SUMB_THREADS = 1024;
constexpr int SUMB_MAX = SB_THREADS;  // workgroups: a pair for each thread of the second launch
constexpr int SUMB_V = 4;             // float4s in flight per thread
// row length + rows (the length of the chain) from which on the pass and its launch
// pay for themselves: 16 x 400 6.6 us both ways, 128 x 256 6.7 -> 6.9, 256 x 256 7.4 ->
// 6.7, 16 x 512 7.3 -> 6.7
constexpr int SUMB_MIN = 512;
struct SumPair {
    double s, a;
};
constexpr size_t SUMB_BYTES = SUMB_MAX * sizeof(SumPair);

// the pair of all WAVES waves' lanes, in every thread (sh: one pair per wave)
template <int WAVES>
__device__ __forceinline__ SumPair sum_pair_all(SumPair v, SumPair* sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        v.s += __shfl_xor(v.s, o);
        v.a += __shfl_xor(v.a, o);
    }
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    SumPair t = sh[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        t.s += sh[w].s;
        t.a += sh[w].a;
    }
    __syncthreads();
    return t;
}

// pairs[workgroup] = the sum and the sum of magnitudes of its share of n floats. The
// float4s begin at the first 16-byte boundary; what lies before and after them goes
// to the first threads of workgroup 0.
__global__ __launch_bounds__(SUMB_THREADS) void k_sum_bounded(const float* __restrict__ a, int64_t n,
                                                              SumPair* __restrict__ pairs) {
    __shared__ SumPair sh[SUMB_THREADS / 64];
    const int64_t pre = (int64_t) ((16u - (uint32_t) ((uintptr_t) a & 15u)) & 15u) / 4;
    const int64_t head = pre < n ? pre : n;
    const int64_t n4 = (n - head) / 4;
    const f4* v = (const f4*) (a + head);
    double s[4] = {0.0, 0.0, 0.0, 0.0}, m[4] = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](int k, float x) {
        const double e = (double) x;
        s[k] += e;
        m[k] += __builtin_fabs(e);
    };
    const int64_t stride = (int64_t) gridDim.x * SUMB_THREADS;
    int64_t i = (int64_t) blockIdx.x * SUMB_THREADS + threadIdx.x;
    for (; i + (SUMB_V - 1) * stride < n4; i += SUMB_V * stride) {
        f4 q[SUMB_V];
#pragma unroll
        for (int u = 0; u < SUMB_V; ++u) q[u] = v[i + u * stride];
#pragma unroll
        for (int u = 0; u < SUMB_V; ++u)
#pragma unroll
            for (int k = 0; k < 4; ++k) add(k, q[u][k]);
    }
    for (; i < n4; i += stride) {
        const f4 q = v[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) add(k, q[k]);
    }
    if (blockIdx.x == 0) {
        const int64_t rest = n - head - 4 * n4;  // under 4, as head is
        if ((int64_t) threadIdx.x < head) add(0, a[threadIdx.x]);
        if ((int64_t) threadIdx.x < rest) add(1, a[head + 4 * n4 + threadIdx.x]);
    }
    const SumPair t = sum_pair_all<SUMB_THREADS / 64>({(s[0] + s[1]) + (s[2] + s[3]), (m[0] + m[1]) + (m[2] + m[3])}, sh);
    if (threadIdx.x == 0) pairs[blockIdx.x] = t;
}

struct SumCheck {
    const SumPair* pairs;
    int n;         // of them
    double rel;    // b / A
};

template <bool VEC, bool CHECKED>
__global__ __launch_bounds__(SB_THREADS) void k_sum_rows_lds(const uint8_t* __restrict__ a, Shape4 sa, double* part,
                                                             uint32_t* ticket, float* __restrict__ d, SumCheck chk) {
    constexpr int W = VEC ? 4 : 1;                         // elements per load
    constexpr int PER = SB_ROWS * SB_C / W / SB_THREADS;   // loads per thread and chunk
    static_assert(PER * SB_THREADS * W == SB_ROWS * SB_C, "a chunk is whole loads per thread");
    static_assert(SB_C / W <= SB_THREADS, "a thread's loads are whole rows apart");
    __shared__ __attribute__((aligned(16))) double ring[SB_RING];
    __shared__ uint32_t order;
    if constexpr (CHECKED) {
        SumPair v = {0.0, 0.0};
        if ((int) threadIdx.x < chk.n) v = chk.pairs[threadIdx.x];
        v = sum_pair_all<SB_THREADS / 64>(v, (SumPair*) ring);
        const double b = chk.rel * v.a;
        const float lo = (float) (v.s - b), hi = (float) (v.s + b);
        if (v.a < __builtin_inf() && __builtin_bit_cast(uint32_t, lo) == __builtin_bit_cast(uint32_t, hi)) {
            if (blockIdx.x == 0 && threadIdx.x == 0) *d = lo;
            return;
        }
    }
    const int64_t rows = sa.ne[1] * sa.ne[2] * sa.ne[3];
    const int64_t r0 = (int64_t) blockIdx.x * SB_ROWS;
    const int64_t n = sa.ne[0];
    const int64_t chunks = (n + SB_C - 1) / SB_C;
    const int tid = threadIdx.x;
    // load u of this thread: row tid / (SB_C / W) + u * (rows a pass covers), the same place in every row
    const int lq = tid % (SB_C / W), lr = tid / (SB_C / W);
    constexpr int STEP = SB_THREADS / (SB_C / W);
    const uint8_t* src[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        int64_t r = r0 + lr + u * STEP;
        r = r < rows ? r : rows - 1;  // rows past the end re-read the last; nobody adds them
        const int64_t i1 = r % sa.ne[1], i2 = (r / sa.ne[1]) % sa.ne[2], i3 = r / (sa.ne[1] * sa.ne[2]);
        src[u] = a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3];
    }
    // elements past the row's end are read from its last ones and staged as zeros
    auto load = [&](int64_t c, float (&v)[PER][W]) {
        const int64_t e = c * SB_C + lq * W;
        const int64_t at = (e < n ? e : n - W) * (VEC ? 4 : sa.nb[0]);
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            if constexpr (VEC) {
                const f4 q = *(const f4*) (src[u] + at);
#pragma unroll
                for (int k = 0; k < 4; ++k) v[u][k] = q[k];
            } else {
                v[u][0] = *(const float*) (src[u] + at);
            }
        }
    };
    auto store = [&](int64_t c, const float (&v)[PER][W]) {
        double* slot = ring + (int) (c % SB_D) * SB_ROWS * SB_LD;
        const bool in = c * SB_C + lq * W < n;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            double* o = slot + (lr + u * STEP) * SB_LD + W * lq;
            if constexpr (VEC) {
                *(sb_d2*) o = sb_d2{in ? (double) v[u][0] : 0.0, in ? (double) v[u][1] : 0.0};
                *(sb_d2*) (o + 2) = sb_d2{in ? (double) v[u][2] : 0.0, in ? (double) v[u][3] : 0.0};
            } else {
                *o = in ? (double) v[u][0] : 0.0;
            }
        }
    };
    for (int64_t c = 0; c < SB_D - 1 && c < chunks; ++c) {
        float v[PER][W];
        load(c, v);
        store(c, v);
    }
    __syncthreads();
    double s = 0.0;
    const bool chain = tid < SB_ROWS && r0 + tid < rows;
    for (int64_t c = 0; c < chunks; ++c) {
        float v[PER][W];
        const bool more = c + SB_D - 1 < chunks;
        if (more) load(c + SB_D - 1, v);
        if (chain) {
            const int64_t left = n - c * SB_C;
            s = sum_chain(s, ring + (int) (c % SB_D) * SB_ROWS * SB_LD + tid * SB_LD,
                          left < SB_C ? ((int) left + 15) / 16 * 16 : SB_C);
        }
        __syncthreads();
        if (more) store(c + SB_D - 1, v);
    }
    // the row sums are written through to where every XCD reads them, then counted
    if (tid < 64) {
        if (chain) __hip_atomic_store(part + r0 + tid, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (tid == 0) order = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (order != gridDim.x - 1) return;
    double total = 0.0;
    constexpr int BATCH = SB_RING / 16 * 16;
    for (int64_t b = 0; b < rows; b += BATCH) {
        const int m = (int) (rows - b < BATCH ? rows - b : BATCH), m16 = (m + 15) / 16 * 16;
        for (int k = tid; k < m16; k += SB_THREADS)
            ring[k] = k < m ? __hip_atomic_load(part + b + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
        __syncthreads();
        if (tid == 0) total = sum_chain(total, ring, m16);
        __syncthreads();
    }
    if (tid == 0) {
        *d = (float) total;
        __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
}

// *d = (float) (0 + part[0] + part[1] + ...), in row order. Up to SC_BATCH row
// sums at a time are staged in LDS by the whole wave (all loads in flight
// together), then lane 0 adds them, reading the next pair while adding one.
constexpr int SC_BATCH = 4096;
__global__ __launch_bounds__(64) void k_sum_combine(const double* __restrict__ part, int64_t rows,
                                                    float* __restrict__ d) {
    __shared__ __attribute__((aligned(16))) double buf[SC_BATCH];
    double total = 0.0;
    for (int64_t r0 = 0; r0 < rows; r0 += SC_BATCH) {
        const int n = (int) (rows - r0 < SC_BATCH ? rows - r0 : SC_BATCH);
        for (int k = threadIdx.x; k < n; k += 64) buf[k] = part[r0 + k];
        __syncthreads();
        if (threadIdx.x == 0) {
            int k = 0;
            if (n >= 8) {
                typedef double d2 __attribute__((ext_vector_type(2)));
                d2 cur[4], nxt[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) cur[q] = *(const d2*) (buf + 2 * q);
                for (; k + 8 <= n; k += 8) {
                    const bool more = k + 16 <= n;
#pragma unroll
                    for (int q = 0; q < 4; ++q) nxt[q] = more ? *(const d2*) (buf + k + 8 + 2 * q) : cur[q];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        total = total + cur[q].x;
                        total = total + cur[q].y;
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) cur[q] = nxt[q];
                }
            }
            for (; k < n; ++k) total = total + buf[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *d = (float) total;
}

// The same sums in one workgroup: each thread sums one row of a block of
// SUM_THREADS rows into LDS, then thread 0 adds the block's row sums in order.
constexpr int SUM_THREADS = 1024;
__global__ __launch_bounds__(SUM_THREADS) void k_sum(const uint8_t* __restrict__ a, Shape4 sa, float* __restrict__ d) {
    __shared__ double row[SUM_THREADS];
    const int64_t rows = sa.ne[1] * sa.ne[2] * sa.ne[3];
    double total = 0.0;
    for (int64_t r0 = 0; r0 < rows; r0 += SUM_THREADS) {
        const int64_t r = r0 + threadIdx.x;
        double s = 0.0;
        if (r < rows) {
            const int64_t i1 = r % sa.ne[1], i2 = (r / sa.ne[1]) % sa.ne[2], i3 = r / (sa.ne[1] * sa.ne[2]);
            const uint8_t* p = a + i1 * sa.nb[1] + i2 * sa.nb[2] + i3 * sa.nb[3];
            for (int64_t i0 = 0; i0 < sa.ne[0]; ++i0) s = s + (double) *(const float*) (p + i0 * sa.nb[0]);
        }
        row[threadIdx.x] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int64_t n = rows - r0 < SUM_THREADS ? rows - r0 : SUM_THREADS;
            for (int64_t k = 0; k < n; ++k) total = total + row[k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *d = (float) total;
}

// contiguous copy of n floats (acc with inplace == false starts from a)
__global__ __launch_bounds__(EW_THREADS) void k_copy_f32(const float* __restrict__ src, float* __restrict__ dst,
                                                         int64_t n) {
    for (int64_t i = (int64_t) blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += (int64_t) gridDim.x * EW_THREADS) {
        dst[i] = src[i];
    }
}

// d[offset + i0*4 + i1*nb1 + i2*nb2 + i3*nb3] += b[i]; the launcher has checked
// that no two elements of b land on the same float, so rows run in parallel
__global__ __launch_bounds__(EW_THREADS) void k_acc(const uint8_t* __restrict__ b, Shape4 sb, uint8_t* __restrict__ d,
                                                    int64_t offset, int64_t nb1, int64_t nb2, int64_t nb3) {
    const int64_t rows = sb.ne[1] * sb.ne[2] * sb.ne[3];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sb.ne[1], i2 = (r / sb.ne[1]) % sb.ne[2], i3 = r / (sb.ne[1] * sb.ne[2]);
        const uint8_t* pb = b + i1 * sb.nb[1] + i2 * sb.nb[2] + i3 * sb.nb[3];
        uint8_t* pd = d + offset + i1 * nb1 + i2 * nb2 + i3 * nb3;
        for (int64_t i0 = threadIdx.x; i0 < sb.ne[0]; i0 += EW_THREADS) {
            float* t = (float*) (pd + i0 * 4);
            *t = *t + *(const float*) (pb + i0 * sb.nb[0]);
        }
    }
}

// k_acc with four floats per lane: rows of b and of the region 16-byte aligned, ne0 a
// multiple of 4 ([4096, 512]: 7.5 -> 5.5 us; where the region is one run, k_flat does
// as well)
__global__ __launch_bounds__(EW_THREADS) void k_acc4(const uint8_t* __restrict__ b, Shape4 sb, uint8_t* __restrict__ d,
                                                     int64_t offset, int64_t nb1, int64_t nb2, int64_t nb3) {
    const int64_t rows = sb.ne[1] * sb.ne[2] * sb.ne[3];
    const int64_t n4 = sb.ne[0] / 4;
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const int64_t i1 = r % sb.ne[1], i2 = (r / sb.ne[1]) % sb.ne[2], i3 = r / (sb.ne[1] * sb.ne[2]);
        const f4* pb = (const f4*) (b + i1 * sb.nb[1] + i2 * sb.nb[2] + i3 * sb.nb[3]);
        f4* pd = (f4*) (d + offset + i1 * nb1 + i2 * nb2 + i3 * nb3);
        for (int64_t q = threadIdx.x; q < n4; q += EW_THREADS) pd[q] = pd[q] + pb[q];
    }
}

// d (contiguous, shape dn) = sum over the repeats of a; every output is summed
// from 0 in a's linear element order: repeat index k3, k2, k1, k0, k0 fastest
__global__ __launch_bounds__(EW_THREADS) void k_repeat_back(const uint8_t* __restrict__ a, Shape4 sa,
                                                            float* __restrict__ d, Shape4 sd) {
    const int64_t n = sd.ne[0] * sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int64_t r0 = sa.ne[0] / sd.ne[0], r1 = sa.ne[1] / sd.ne[1], r2 = sa.ne[2] / sd.ne[2],
                  r3 = sa.ne[3] / sd.ne[3];
    for (int64_t j = (int64_t) blockIdx.x * EW_THREADS + threadIdx.x; j < n; j += (int64_t) gridDim.x * EW_THREADS) {
        const int64_t j0 = j % sd.ne[0], j1 = (j / sd.ne[0]) % sd.ne[1], j2 = (j / (sd.ne[0] * sd.ne[1])) % sd.ne[2],
                      j3 = j / (sd.ne[0] * sd.ne[1] * sd.ne[2]);
        float s = 0.f;
        for (int64_t k3 = 0; k3 < r3; ++k3)
            for (int64_t k2 = 0; k2 < r2; ++k2)
                for (int64_t k1 = 0; k1 < r1; ++k1) {
                    const uint8_t* row = a + (j1 + k1 * sd.ne[1]) * sa.nb[1] + (j2 + k2 * sd.ne[2]) * sa.nb[2] +
                                         (j3 + k3 * sd.ne[3]) * sa.nb[3];
                    for (int64_t k0 = 0; k0 < r0; ++k0) s = s + *(const float*) (row + (j0 + k0 * sd.ne[0]) * sa.nb[0]);
                }
        d[j] = s;
    }
}

// The same sums when ne0 is not repeated (a.ne0 == d.ne0, e.g. a bias gradient
// summed over the tokens): output j's terms are rows k1, k2, k3 (k1 fastest) at
// one column, so their offsets from a's element j follow a counter that is the
// same for every lane. RB_AHEAD loads run ahead of the in-order adds, from
// offsets that stay inside a (terms past the last re-read the first).
constexpr int RB_THREADS = 64;
constexpr int RB_AHEAD = 64;
__global__ __launch_bounds__(RB_THREADS) void k_repeat_back_cols(const uint8_t* __restrict__ a, Shape4 sa,
                                                                 float* __restrict__ d, Shape4 sd) {
    const int64_t n = sd.ne[0] * sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int64_t j = (int64_t) blockIdx.x * RB_THREADS + threadIdx.x;
    if (j >= n) return;  // no barrier below
    const int64_t j0 = j % sd.ne[0], j1 = (j / sd.ne[0]) % sd.ne[1], j2 = (j / (sd.ne[0] * sd.ne[1])) % sd.ne[2],
                  j3 = j / (sd.ne[0] * sd.ne[1] * sd.ne[2]);
    const uint8_t* base = a + j0 * sa.nb[0] + j1 * sa.nb[1] + j2 * sa.nb[2] + j3 * sa.nb[3];
    const int64_t r1 = sa.ne[1] / sd.ne[1], r2 = sa.ne[2] / sd.ne[2], r3 = sa.ne[3] / sd.ne[3];
    const int64_t st1 = sd.ne[1] * sa.nb[1], st2 = sd.ne[2] * sa.nb[2], st3 = sd.ne[3] * sa.nb[3];
    const int64_t terms = r1 * r2 * r3;
    // the counter of the next term to load: (k1, k2, k3) and its byte offset
    int64_t k1 = 0, k2 = 0, k3 = 0, off = 0, next = 0;
    auto advance = [&]() {
        ++next;
        ++k1;
        off += st1;
        if (k1 == r1) {
            k1 = 0;
            off -= r1 * st1;
            ++k2;
            off += st2;
            if (k2 == r2) {
                k2 = 0;
                off -= r2 * st2;
                ++k3;
                off += st3;
            }
        }
    };
    float buf[RB_AHEAD];
#pragma unroll
    for (int u = 0; u < RB_AHEAD; ++u) {
        buf[u] = *(const float*) (base + (next < terms ? off : 0));
        advance();
    }
    float s = 0.f;
    for (int64_t q0 = 0; q0 < terms; q0 += RB_AHEAD) {
#pragma unroll
        for (int u = 0; u < RB_AHEAD; ++u) {
            if (q0 + u < terms) s = s + buf[u];  // the same for every lane
            buf[u] = *(const float*) (base + (next < terms ? off : 0));
            advance();
        }
    }
    d[j] = s;
}

// k_repeat_back_cols when only dim 1 repeats (output j's terms are a's element j
// and every st1 bytes after it), with the loads spread over a workgroup: O
// consecutive outputs per workgroup, T terms of each per chunk, streamed through an
// LDS ring of D chunks by all RL_THREADS threads, D - 1 chunks ahead of wave 0, whose
// lane o adds output o's terms in order. The first D - 1 chunks are asked for
// together; each later one waits for its loads alone. So while few outputs leave
// CUs idle, workgroups take 16 of them and long chunks (bound by the loads' latency:
// 64 outputs and 32 terms -> 16 and 128: 4096 outputs of 512 terms 10.3 -> 6.8 us, 777
// of 130 4.9 -> 3.9, 100 of 8192 128 -> 76); more outputs take 64, whole lines of
// 256 bytes (16384 of 512 10.7 us, with 16 at a time 14.7).
constexpr int RL_THREADS = 256;
constexpr int RL_MIN = 64;       // terms from which on
constexpr int RL_AT_ONCE = 32;   // terms read from LDS ahead of their adds
template <int RL_O, int RL_T, int RL_D>
__global__ __launch_bounds__(RL_THREADS) void k_repeat_back_lds(const uint8_t* __restrict__ a, Shape4 sa,
                                                                float* __restrict__ d, Shape4 sd) {
    constexpr int RL_STEP = RL_THREADS / RL_O;  // terms between two loads of a thread
    constexpr int RL_PER = RL_T / RL_STEP;      // loads per thread and chunk
    static_assert(RL_THREADS % RL_O == 0 && RL_O <= 64, "a thread loads one output's terms, wave 0 adds them");
    static_assert(RL_T % RL_STEP == 0 && RL_T % RL_AT_ONCE == 0 && RL_D >= 3, "whole loads; one barrier per chunk");
    __shared__ float ring[RL_D * RL_T * RL_O];
    const int64_t n = sd.ne[0] * sd.ne[1] * sd.ne[2] * sd.ne[3];
    const int tid = threadIdx.x, o = tid % RL_O;
    int64_t j = (int64_t) blockIdx.x * RL_O + o;
    const bool valid = j < n;
    j = valid ? j : n - 1;  // outputs past the end re-read the last; nobody stores them
    const int64_t j0 = j % sd.ne[0], j1 = (j / sd.ne[0]) % sd.ne[1], j2 = (j / (sd.ne[0] * sd.ne[1])) % sd.ne[2],
                  j3 = j / (sd.ne[0] * sd.ne[1] * sd.ne[2]);
    const uint8_t* base = a + j0 * sa.nb[0] + j1 * sa.nb[1] + j2 * sa.nb[2] + j3 * sa.nb[3];
    const int64_t terms = sa.ne[1] / sd.ne[1];
    const int64_t st1 = sd.ne[1] * sa.nb[1];
    const int64_t chunks = (terms + RL_T - 1) / RL_T;
    auto load = [&](int64_t c, float (&v)[RL_PER]) {
#pragma unroll
        for (int u = 0; u < RL_PER; ++u) {
            const int64_t q = c * RL_T + tid / RL_O + RL_STEP * u;  // this load's term
            v[u] = *(const float*) (base + (q < terms ? q : terms - 1) * st1);
        }
    };
    auto store = [&](int64_t c, const float (&v)[RL_PER]) {
        float* slot = ring + (int) (c % RL_D) * RL_T * RL_O;
#pragma unroll
        for (int u = 0; u < RL_PER; ++u) slot[tid + RL_THREADS * u] = v[u];  // [term][output]
    };
    // (chunks past the last are its last term again, and nobody adds them)
    float first[RL_D - 1][RL_PER];
#pragma unroll
    for (int c = 0; c < RL_D - 1; ++c) load(c, first[c]);
#pragma unroll
    for (int c = 0; c < RL_D - 1; ++c) store(c, first[c]);
    __syncthreads();
    float s = 0.f;
    for (int64_t c = 0; c < chunks; ++c) {
        float v[RL_PER];
        const bool more = c + RL_D - 1 < chunks;
        if (more) load(c + RL_D - 1, v);
        if (tid < RL_O) {
            const float* slot = ring + (int) (c % RL_D) * RL_T * RL_O + o;
            const int m = (int) (terms - c * RL_T < RL_T ? terms - c * RL_T : RL_T);
            int q0 = 0;
            for (; q0 + RL_AT_ONCE <= m; q0 += RL_AT_ONCE) {  // read together, then added in order
                float t[RL_AT_ONCE];
#pragma unroll
                for (int q = 0; q < RL_AT_ONCE; ++q) t[q] = slot[(q0 + q) * RL_O];
#pragma unroll
                for (int q = 0; q < RL_AT_ONCE; ++q) s = s + t[q];
            }
            for (; q0 < m; ++q0) s = s + slot[q0 * RL_O];
        }
        __syncthreads();
        if (more) store(c + RL_D - 1, v);
    }
    if (tid < RL_O && valid) d[j] = s;
}

// The same sums when ne0 is not repeated and each has few terms (the gradient of a
// broadcast operand, summed over the planes that shared it): one output, or four
// along ne0 (VEC: rows of both 16-byte aligned), per lane, RF_AHEAD terms loaded
// ahead of the in-order adds. Bound by HBM; k_repeat_back_cols asks for 128 terms
// whatever their number ([64, 333, 12, 2] to 4 planes of the 12: 21.5 -> 4.4 us).
constexpr int RF_AHEAD = 4;
template <bool VEC>
__global__ __launch_bounds__(EW_THREADS) void k_repeat_back_few(const uint8_t* __restrict__ a, Shape4 sa,
                                                                float* __restrict__ d, uint32_t n, FastDiv ne0,
                                                                FastDiv ne1, FastDiv ne2, int r1, int r2, int r3) {
    constexpr int W = VEC ? 4 : 1;
    const uint32_t j = blockIdx.x * EW_THREADS + threadIdx.x;
    if (j >= n) return;  // no barrier below
    const uint32_t q1 = div_by(j, ne0), j0 = j - q1 * ne0.d;
    const uint32_t q2 = div_by(q1, ne1), j1 = q1 - q2 * ne1.d;
    const uint32_t j3 = div_by(q2, ne2), j2 = q2 - j3 * ne2.d;
    const uint8_t* base = a + (int64_t) j0 * W * sa.nb[0] + j1 * sa.nb[1] + j2 * sa.nb[2] + j3 * sa.nb[3];
    const int64_t st1 = ne1.d * sa.nb[1], st2 = ne2.d * sa.nb[2], st3 = (sa.ne[3] / r3) * sa.nb[3];
    const int terms = r1 * r2 * r3;
    // the next term to load, k1 fastest, and its offset
    int k1 = 0, k2 = 0, k3 = 0, next = 0;
    auto fetch = [&](float (&v)[W]) {
        const uint8_t* p = base + (next < terms ? k1 * st1 + k2 * st2 + k3 * st3 : 0);
        if constexpr (VEC) {
            const f4 q = *(const f4*) p;
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = q[c];
        } else {
            v[0] = *(const float*) p;
        }
        ++next;
        if (++k1 == r1) {
            k1 = 0;
            if (++k2 == r2) {
                k2 = 0;
                ++k3;
            }
        }
    };
    float s[W];
#pragma unroll
    for (int c = 0; c < W; ++c) s[c] = 0.f;
    for (int t = 0; t < terms; t += RF_AHEAD) {
        float v[RF_AHEAD][W];
#pragma unroll
        for (int u = 0; u < RF_AHEAD; ++u) fetch(v[u]);
#pragma unroll
        for (int u = 0; u < RF_AHEAD; ++u) {
            if (t + u < terms) {  // the same for every lane
#pragma unroll
                for (int c = 0; c < W; ++c) s[c] = s[c] + v[u][c];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < W; ++c) d[(int64_t) j * W + c] = s[c];
}

unsigned grid_for(int64_t work, int64_t per_block) {
    int64_t g = (work + per_block - 1) / per_block;
    const int64_t cap = (int64_t) device_cus() * 16;
    if (g > cap) g = cap;
    return (unsigned) (g < 1 ? 1 : g);
}

bool f32_aligned(const trc_hip_tensor& t) {
    if ((((uintptr_t) t.data) & 3u) != 0) return false;
    for (int d = 0; d < 4; ++d) {
        if ((t.nb[d] & 3u) != 0) return false;
    }
    return true;
}

bool contiguous_f32(const trc_hip_tensor& t) {
    size_t nb = 4;
    for (int d = 0; d < 4; ++d) {
        if (t.ne[d] > 1 && t.nb[d] != nb) return false;
        nb *= (size_t) t.ne[d];
    }
    return true;
}

int64_t nelem(const trc_hip_tensor& t) { return t.ne[0] * t.ne[1] * t.ne[2] * t.ne[3]; }

// Every row (ne0-run) starts 16-byte aligned and holds whole float4s.
bool rows_vec4(const trc_hip_tensor& t) {
    if (t.nb[0] != 4 || t.ne[0] % 4 != 0 || (((uintptr_t) t.data) & 15u) != 0) return false;
    for (int d = 1; d < 4; ++d) {
        if (t.ne[d] > 1 && t.nb[d] % 16 != 0) return false;
    }
    return true;
}

bool shape_ok(const trc_hip_tensor& t) {
    for (int d = 0; d < 4; ++d) {
        if (t.ne[d] <= 0) return false;
    }
    return true;
}

bool flat_f32(const trc_hip_tensor& t) { return (((uintptr_t) t.data) & 15u) == 0 && contiguous_f32(t); }

constexpr int64_t FLAT_MAX = (int64_t) 1 << 33;  // floats of a launch
static_assert(FLAT_MAX / 4 / EW_THREADS < max_groups(EW_THREADS), "under 2^32 threads");
template <FlatOp OP>
int launch_flat(const char* name, const void* a, const void* b, void* d, int64_t n, float scale, hipStream_t s) {
    for (int64_t at = 0; at < n; at += FLAT_MAX) {
        const int64_t m = n - at < FLAT_MAX ? n - at : FLAT_MAX;
        const int64_t blocks = (m / 4 + EW_THREADS) / EW_THREADS;  // one more float4 for the tail
        const f4* fa = (const f4*) ((const float*) a + at);
        const f4* fb = b != nullptr ? (const f4*) ((const float*) b + at) : nullptr;
        f4* fd = (f4*) ((float*) d + at);
        if (n >= FLAT_NT) {
            hipLaunchKernelGGL((k_flat<OP, true>), dim3((unsigned) blocks), dim3(EW_THREADS), 0, s, fa, fb, fd, m, scale);
        } else {
            hipLaunchKernelGGL((k_flat<OP, false>), dim3((unsigned) blocks), dim3(EW_THREADS), 0, s, fa, fb, fd, m, scale);
        }
        const int rc = check_launch(name);
        if (rc != TRC_HIP_OK) return rc;
    }
    return TRC_HIP_OK;
}

template <BinOp OP>
int launch_binary(const char* name, const trc_hip_tensor& a, const trc_hip_tensor& b, const trc_hip_tensor& d,
                  hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || b.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) {
        return fail(TRC_HIP_E_INVALID, "%s: F32 tensors only", name);
    }
    if (!shape_ok(a) || !shape_ok(b) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "%s: empty or negative extent", name);
    for (int k = 0; k < 4; ++k) {
        if (d.ne[k] != a.ne[k] || (b.ne[k] != a.ne[k] && b.ne[k] != 1)) {
            return fail(TRC_HIP_E_SHAPE, "%s: dst must have a's shape and b must broadcast to it (dim %d)", name, k);
        }
    }
    if (!f32_aligned(a) || !f32_aligned(b) || !f32_aligned(d)) return fail(TRC_HIP_E_ALIGN, "%s: 4-byte alignment", name);
    if (flat_f32(a) && flat_f32(d) && flat_f32(b) && nelem(a) == nelem(b)) {
        return launch_flat<OP == BinOp::ADD ? FlatOp::ADD : FlatOp::MUL>(name, a.data, b.data, d.data, nelem(d), 0.f, s);
    }
    const int64_t rows = d.ne[1] * d.ne[2] * d.ne[3];
    if (rows_vec4(a) && rows_vec4(d) && (b.ne[0] == 1 || rows_vec4(b))) {
        hipLaunchKernelGGL(k_binary4<OP>, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                           shape_of(a), (const uint8_t*) b.data, shape_of(b), (uint8_t*) d.data, shape_of(d));
        return check_launch(name);
    }
    hipLaunchKernelGGL(k_binary<OP>, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                       shape_of(a), (const uint8_t*) b.data, shape_of(b), (uint8_t*) d.data, shape_of(d));
    return check_launch(name);
}

}  // namespace

int launch_add_f32(const trc_hip_tensor& a, const trc_hip_tensor& b, const trc_hip_tensor& d, hipStream_t s) {
    return launch_binary<BinOp::ADD>("add", a, b, d, s);
}

int launch_mul_f32(const trc_hip_tensor& a, const trc_hip_tensor& b, const trc_hip_tensor& d, hipStream_t s) {
    return launch_binary<BinOp::MUL>("mul", a, b, d, s);
}

namespace {

template <UnOp OP>
int launch_unary(const char* name, const trc_hip_tensor& a, const trc_hip_tensor& d, float scale, hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) return fail(TRC_HIP_E_INVALID, "%s: F32 tensors only", name);
    if (!shape_ok(a) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "%s: empty or negative extent", name);
    for (int k = 0; k < 4; ++k) {
        if (d.ne[k] != a.ne[k]) return fail(TRC_HIP_E_SHAPE, "%s: dst must have a's shape (dim %d)", name, k);
    }
    if (!f32_aligned(a) || !f32_aligned(d)) return fail(TRC_HIP_E_ALIGN, "%s: 4-byte alignment", name);
    if (flat_f32(a) && flat_f32(d)) {
        return launch_flat<OP == UnOp::SQR ? FlatOp::SQR : FlatOp::SCALE>(name, a.data, nullptr, d.data, nelem(d), scale, s);
    }
    const int64_t rows = d.ne[1] * d.ne[2] * d.ne[3];
    if (rows_vec4(a) && rows_vec4(d)) {
        hipLaunchKernelGGL(k_unary4<OP>, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                           shape_of(a), (uint8_t*) d.data, shape_of(d), scale);
        return check_launch(name);
    }
    hipLaunchKernelGGL(k_unary<OP>, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                       shape_of(a), (uint8_t*) d.data, shape_of(d), scale);
    return check_launch(name);
}

}  // namespace

int launch_sqr_f32(const trc_hip_tensor& a, const trc_hip_tensor& d, hipStream_t s) {
    return launch_unary<UnOp::SQR>("sqr", a, d, 0.f, s);
}

int launch_scale_f32(const trc_hip_tensor& a, const trc_hip_tensor& d, float scale, hipStream_t s) {
    return launch_unary<UnOp::SCALE>("scale", a, d, scale, s);
}

int launch_repeat_f32(const trc_hip_tensor& a, const trc_hip_tensor& d, hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) return fail(TRC_HIP_E_INVALID, "repeat: F32 tensors only");
    if (!shape_ok(a) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "repeat: empty or negative extent");
    for (int k = 0; k < 4; ++k) {
        // ggml_can_repeat(a, dst): every dst extent a multiple of a's
        if (d.ne[k] % a.ne[k] != 0) return fail(TRC_HIP_E_SHAPE, "repeat: dst.ne[%d] is not a multiple of a.ne[%d]", k, k);
    }
    if (!f32_aligned(a) || !f32_aligned(d)) return fail(TRC_HIP_E_ALIGN, "repeat: 4-byte alignment");
    const int64_t n = nelem(d);
    if (rows_vec4(d)) {
        const int64_t rows = d.ne[1] * d.ne[2] * d.ne[3];
        hipLaunchKernelGGL(k_repeat4, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                           shape_of(a), (uint8_t*) d.data, shape_of(d));
        return check_launch("repeat");
    }
    hipLaunchKernelGGL(k_repeat, dim3(grid_for(n, EW_THREADS)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                       shape_of(a), (uint8_t*) d.data, shape_of(d));
    return check_launch("repeat");
}

int launch_sum_f32(const trc_hip_tensor& a, const trc_hip_tensor& d, hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) return fail(TRC_HIP_E_INVALID, "sum: F32 tensors only");
    if (!shape_ok(a) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "sum: empty or negative extent");
    if (nelem(d) != 1) return fail(TRC_HIP_E_SHAPE, "sum: dst must hold one element");
    if (!f32_aligned(a) || !f32_aligned(d)) return fail(TRC_HIP_E_ALIGN, "sum: 4-byte alignment");
    const int64_t rows = a.ne[1] * a.ne[2] * a.ne[3];
    if ((size_t) rows * sizeof(double) > qm_workspace_bytes()) {
        hipLaunchKernelGGL(k_sum, dim3(1), dim3(SUM_THREADS), 0, s, (const uint8_t*) a.data, shape_of(a),
                           (float*) d.data);
        return check_launch("sum");
    }
    // the row sums go to this stream's workspace (the one trc_hip_qmatvec uses;
    // work on one stream runs in order, so the two never meet)
    uint8_t* ws = nullptr;
    const int rc = qm_stream_workspace(s, &ws);
    if (rc != TRC_HIP_OK) return rc;
    const bool vec = a.nb[0] == 4 && (((uintptr_t) a.data) & 15u) == 0 && (a.ne[1] == 1 || a.nb[1] % 16 == 0) &&
                     (a.ne[2] == 1 || a.nb[2] % 16 == 0) && (a.ne[3] == 1 || a.nb[3] % 16 == 0);
    const unsigned grid = (unsigned) ((rows + SR_THREADS - 1) / SR_THREADS);
    if (a.ne[0] >= SB_MIN) {
        uint32_t* ticket = (uint32_t*) (ws + qm_workspace_bytes());
        const dim3 g((unsigned) ((rows + SB_ROWS - 1) / SB_ROWS));
        const bool whole = vec && a.ne[0] % 4 == 0;
        const int64_t n = rows * a.ne[0];
        const bool run = a.nb[0] == 4 && (a.ne[1] == 1 || (int64_t) a.nb[1] == 4 * a.ne[0]) &&
                         (a.ne[2] == 1 || (int64_t) a.nb[2] == 4 * a.ne[0] * a.ne[1]) &&
                         (a.ne[3] == 1 || (int64_t) a.nb[3] == 4 * a.ne[0] * a.ne[1] * a.ne[2]);
        SumCheck chk = {nullptr, 0, 0.0};
        if (run && a.ne[0] + rows >= SUMB_MIN && (size_t) rows * sizeof(double) + SUMB_BYTES <= qm_workspace_bytes()) {
            SumPair* pairs = (SumPair*) (ws + qm_workspace_bytes() - SUMB_BYTES);
            const int64_t want = (n + 4 * SUMB_THREADS - 1) / (4 * SUMB_THREADS);
            chk.pairs = pairs;
            chk.n = (int) (want < SUMB_MAX ? want : SUMB_MAX);
            // roundings on the way of an element: the rows and the row sums; here a
            // thread's, a workgroup's (2 + 6 + 15) and the pairs' (6 + 3); the check's
            const double k = (double) a.ne[0] + (double) rows + (double) n / ((double) chk.n * SUMB_THREADS) + 64.0;
            chk.rel = 1.01 * k * 0x1p-53;
            hipLaunchKernelGGL(k_sum_bounded, dim3((unsigned) chk.n), dim3(SUMB_THREADS), 0, s, (const float*) a.data, n,
                               pairs);
            const int st = check_launch("sum (in any order)");
            if (st != TRC_HIP_OK) return st;
        }
#define TRC_SUM(V, C)                                                                                              \
    hipLaunchKernelGGL((k_sum_rows_lds<V, C>), g, dim3(SB_THREADS), 0, s, (const uint8_t*) a.data, shape_of(a), \
                       (double*) ws, ticket, (float*) d.data, chk)
        if (whole) {
            if (chk.n) TRC_SUM(true, true);
            else TRC_SUM(true, false);
        } else {
            if (chk.n) TRC_SUM(false, true);
            else TRC_SUM(false, false);
        }
#undef TRC_SUM
        return check_launch("sum");
    }
    if (vec) {
        hipLaunchKernelGGL(k_sum_rows<true>, dim3(grid), dim3(SR_THREADS), 0, s, (const uint8_t*) a.data, shape_of(a),
                           (double*) ws);
    } else {
        hipLaunchKernelGGL(k_sum_rows<false>, dim3(grid), dim3(SR_THREADS), 0, s, (const uint8_t*) a.data,
                           shape_of(a), (double*) ws);
    }
    int st = check_launch("sum (rows)");
    if (st != TRC_HIP_OK) return st;
    hipLaunchKernelGGL(k_sum_combine, dim3(1), dim3(64), 0, s, (const double*) ws, rows, (float*) d.data);
    return check_launch("sum (row sums)");
}

int launch_acc_f32(const trc_hip_tensor& a, const trc_hip_tensor& b, const trc_hip_tensor& d, size_t nb1, size_t nb2,
                   size_t nb3, size_t offset, int inplace, hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || b.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) {
        return fail(TRC_HIP_E_INVALID, "acc: F32 tensors only");
    }
    if (!shape_ok(a) || !shape_ok(b) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "acc: empty or negative extent");
    for (int k = 0; k < 4; ++k) {
        if (d.ne[k] != a.ne[k]) return fail(TRC_HIP_E_SHAPE, "acc: dst must have a's shape");
    }
    if (!contiguous_f32(a) || !contiguous_f32(d)) return fail(TRC_HIP_E_SHAPE, "acc: a and dst must be contiguous");
    if (!f32_aligned(a) || !f32_aligned(b) || !f32_aligned(d) || (nb1 & 3u) || (nb2 & 3u) || (nb3 & 3u) ||
        (offset & 3u)) {
        return fail(TRC_HIP_E_ALIGN, "acc: 4-byte alignment of pointers, strides and offset");
    }
    // region inside a (src/core/trc_tensor.cpp:331-337)
    const size_t nbytes = (size_t) nelem(a) * 4;
    size_t last = (size_t) (b.ne[0] - 1) * 4;
    last += b.ne[1] > 1 ? (size_t) (b.ne[1] - 1) * nb1 : 0;
    last += b.ne[2] > 1 ? (size_t) (b.ne[2] - 1) * nb2 : 0;
    last += b.ne[3] > 1 ? (size_t) (b.ne[3] - 1) * nb3 : 0;
    if (offset + last + 4 > nbytes) return fail(TRC_HIP_E_SHAPE, "acc: region leaves the target");
    // the region must not overlap itself: with its dims sorted by stride, each
    // stride must clear the span of the smaller ones
    {
        int64_t ne[4] = {b.ne[0], b.ne[1], b.ne[2], b.ne[3]};
        size_t st[4] = {4, nb1, nb2, nb3};
        int idx[4] = {0, 1, 2, 3};
        for (int i = 1; i < 4; ++i)
            for (int j = i; j > 0 && st[idx[j]] < st[idx[j - 1]]; --j) {
                const int t = idx[j];
                idx[j] = idx[j - 1];
                idx[j - 1] = t;
            }
        size_t span = 0;  // bytes covered by the dims already placed
        for (int i = 0; i < 4; ++i) {
            const int k = idx[i];
            if (ne[k] == 1) continue;
            if (st[k] < (span == 0 ? 4 : span)) return fail(TRC_HIP_E_SHAPE, "acc: region overlaps itself");
            span = st[k] * (size_t) (ne[k] - 1) + (span == 0 ? 4 : span);
        }
    }
    if (!inplace && a.data != d.data) {
        const int64_t n = nelem(a);
        hipLaunchKernelGGL(k_copy_f32, dim3(grid_for(n, EW_THREADS)), dim3(EW_THREADS), 0, s, (const float*) a.data,
                           (float*) d.data, n);
        const int rc = check_launch("acc copy");
        if (rc != TRC_HIP_OK) return rc;
    }
    const int64_t rows = b.ne[1] * b.ne[2] * b.ne[3];
    // a region as dense as b: one run of floats
    if (flat_f32(b) && ((((uintptr_t) d.data) | offset) & 15u) == 0 && (b.ne[1] == 1 || nb1 == (size_t) b.ne[0] * 4) &&
        (b.ne[2] == 1 || nb2 == (size_t) (b.ne[0] * b.ne[1]) * 4) &&
        (b.ne[3] == 1 || nb3 == (size_t) (b.ne[0] * b.ne[1] * b.ne[2]) * 4)) {
        uint8_t* at = (uint8_t*) d.data + offset;
        return launch_flat<FlatOp::ADD>("acc", at, b.data, at, nelem(b), 0.f, s);
    }
    if (rows_vec4(b) && ((((uintptr_t) d.data) | offset) & 15u) == 0 && (b.ne[1] == 1 || nb1 % 16 == 0) &&
        (b.ne[2] == 1 || nb2 % 16 == 0) && (b.ne[3] == 1 || nb3 % 16 == 0)) {
        hipLaunchKernelGGL(k_acc4, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) b.data,
                           shape_of(b), (uint8_t*) d.data, (int64_t) offset, (int64_t) nb1, (int64_t) nb2, (int64_t) nb3);
        return check_launch("acc");
    }
    hipLaunchKernelGGL(k_acc, dim3(grid_for(rows, 1)), dim3(EW_THREADS), 0, s, (const uint8_t*) b.data, shape_of(b),
                       (uint8_t*) d.data, (int64_t) offset, (int64_t) nb1, (int64_t) nb2, (int64_t) nb3);
    return check_launch("acc");
}

int launch_repeat_back_f32(const trc_hip_tensor& a, const trc_hip_tensor& d, hipStream_t s) {
    if (a.type != TRC_HIP_TYPE_F32 || d.type != TRC_HIP_TYPE_F32) {
        return fail(TRC_HIP_E_INVALID, "repeat_back: F32 tensors only");
    }
    if (!shape_ok(a) || !shape_ok(d)) return fail(TRC_HIP_E_SHAPE, "repeat_back: empty or negative extent");
    for (int k = 0; k < 4; ++k) {
        if (a.ne[k] % d.ne[k] != 0) return fail(TRC_HIP_E_SHAPE, "repeat_back: a.ne must be a multiple of dst.ne");
    }
    if (!contiguous_f32(d)) return fail(TRC_HIP_E_SHAPE, "repeat_back: dst must be contiguous");
    if (!f32_aligned(a) || !f32_aligned(d)) return fail(TRC_HIP_E_ALIGN, "repeat_back: 4-byte alignment");
    const int64_t n = nelem(d);
    if (a.ne[0] == d.ne[0] && a.ne[2] == d.ne[2] && a.ne[3] == d.ne[3] && a.ne[1] / d.ne[1] >= RL_MIN) {
        // 16 outputs each while that is at most two workgroups a CU (10240 outputs of
        // 128 terms 4.3 us either way)
        if (n <= 32 * (int64_t) device_cus()) {
            hipLaunchKernelGGL((k_repeat_back_lds<16, 128, 3>), dim3((unsigned) ((n + 15) / 16)), dim3(RL_THREADS), 0, s,
                               (const uint8_t*) a.data, shape_of(a), (float*) d.data, shape_of(d));
        } else {
            hipLaunchKernelGGL((k_repeat_back_lds<64, 32, 4>), dim3((unsigned) ((n + 63) / 64)), dim3(RL_THREADS), 0, s,
                               (const uint8_t*) a.data, shape_of(a), (float*) d.data, shape_of(d));
        }
        return check_launch("repeat_back");
    }
    const int64_t r1 = a.ne[1] / d.ne[1], r2 = a.ne[2] / d.ne[2], r3 = a.ne[3] / d.ne[3];
    // up to RB_AHEAD terms: more keep the pipeline of k_repeat_back_cols busy
    if (a.ne[0] == d.ne[0] && r1 <= RB_AHEAD && r2 <= RB_AHEAD && r3 <= RB_AHEAD && r1 * r2 * r3 <= RB_AHEAD &&
        n < ((int64_t) 1 << 31) - EW_THREADS) {
        const bool vec = rows_vec4(a) && (((uintptr_t) d.data) & 15u) == 0;
        const int64_t units = vec ? n / 4 : n, u0 = vec ? d.ne[0] / 4 : d.ne[0];
        const dim3 grid((unsigned) ((units + EW_THREADS - 1) / EW_THREADS));
        if (vec) {
            hipLaunchKernelGGL(k_repeat_back_few<true>, grid, dim3(EW_THREADS), 0, s, (const uint8_t*) a.data, shape_of(a),
                               (float*) d.data, (uint32_t) units, fast_div(u0), fast_div(d.ne[1]), fast_div(d.ne[2]),
                               (int) r1, (int) r2, (int) r3);
        } else {
            hipLaunchKernelGGL(k_repeat_back_few<false>, grid, dim3(EW_THREADS), 0, s, (const uint8_t*) a.data, shape_of(a),
                               (float*) d.data, (uint32_t) units, fast_div(u0), fast_div(d.ne[1]), fast_div(d.ne[2]),
                               (int) r1, (int) r2, (int) r3);
        }
        return check_launch("repeat_back");
    }
    if (a.ne[0] == d.ne[0]) {
        hipLaunchKernelGGL(k_repeat_back_cols, dim3((unsigned) ((n + RB_THREADS - 1) / RB_THREADS)), dim3(RB_THREADS),
                           0, s, (const uint8_t*) a.data, shape_of(a), (float*) d.data, shape_of(d));
        return check_launch("repeat_back");
    }
    hipLaunchKernelGGL(k_repeat_back, dim3(grid_for(n, EW_THREADS)), dim3(EW_THREADS), 0, s, (const uint8_t*) a.data,
                       shape_of(a), (float*) d.data, shape_of(d));
    return check_launch("repeat_back");
}

}  // namespace trc_hip
