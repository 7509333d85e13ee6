// F32 mul_mat tiles on the bf16 matrix cores, each float held exactly as three
// bf16 (same result rules as mul_mat.hip: compute_mul_mat,
// src/backends/cpu/trc_cpu_ops.cpp:182-216, to rounding).
//
// A float has 24 significant bits, so x = h + m + l with h = bf16(x), m =
// bf16(x - h), l = x - h - m, each of at most 8 bits, and both differences
// exact. The product x y is then the sum of nine bf16 products, each exact in
// the matrix core; the three left out (m l, l m, l l) are under 2^-24 |x y|.
// Six v_mfma_f32_32x32x16_bf16 take 192 cycles of a SIMD for 32 x 32 x 16
// products where v_mfma_f32_32x32x2_f32 takes 512 (and runs at the rate of the
// vector ALU's FMAs). Measured: 4096 x 4096 x 512 89 us, 193 TFLOP/s of F32
// products, the matrix cores busy 52 % of the cycles (FP32 instructions 138 us).
//
// Error against 64 bits: a bf16 instruction rounds its accumulator to nearest once
// per 16 k, so that the error grows with sqrt(K / 16) and, from K = 2 on, stays below
// that of the FP32 instructions, which round at every k (K = 1 does not come here). Rel
// 2-norm, FP32 -> here: normal inputs K = 32 1.05e-7 -> 0.40e-7, 128 1.95e-7 ->
// 0.64e-7, 1024 5.8e-7 -> 1.9e-7, 4096 1.15e-6 -> 0.40e-6, 262144 9.1e-6 -> 2.3e-6;
// uniform in [0, 1) K = 4096 8.4e-7 -> 3.0e-7, 16384 1.7e-6 -> 6.0e-7 with a mean of
// -5e-8, 262144 1.3e-5 -> 1.5e-6. Before it rounds, the instruction drops what lies
// far enough below its accumulator's last bit, downwards; the products are kept apart
// by size for that (below). One kind of input fares worse than on the FP32
// instructions: operands that are all nearly the same number, whose 16-bit first
// products lose the same bits at every rounding (1 + 0.01 u, K = 4096 8.5e-7 -> 3.4e-7,
// but 8192 in one chain 1.2e-6 -> 5.6e-6, 65536 4.5e-6 -> 1.8e-5; at 262144 3.2e-4 ->
// 1.7e-5). A chain is K over the parts, and over two where a tile has 8 waves.
//
// Operands are split as x 2^24 and results scaled back by 2^-48, both exact: every
// part is then 0 or at least 2^-125, a normal bf16, down to the smallest
// subnormal float, so that small values (the tails of a softmax) are held like any
// other. What the split cannot hold is at the other end: x not finite or 2^104 and
// more, or sums from 2^80 on, which leave a result that is not finite. A workgroup
// that finds one repeats its tile with the FP32 instructions, so infinities, NaNs
// and overflows come out as those give them, at the price of both passes: 4096 x
// 4096 x 512 with one infinity 229 us, without 92 (FP32 instructions alone 140).
// (Unscaled, the same repeat was needed for any value under about 2^-110: the
// product with softmax weights of that shape took 238 us, now 92. Nothing that
// would have to be gathered in the loop stays either, and no register spills.)
#pragma once

#include "common.h"
#include "mm_args.h"

#include <type_traits>

namespace trc_hip {
namespace {

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// How the parts of K of a tile come together: a launch of their own each (B3_ALONE:
// K whole, or one part stored or added to dst), in dst through a ticket (B3_PAIR,
// two parts: a + b is the same in either order), or in slots of a workspace that
// the last part to arrive adds up in part order (B3_SLOTS). All three give the
// same bits.
constexpr int B3_ALONE = 0, B3_PAIR = 1, B3_SLOTS = 2;
constexpr int B3_SC1 = 16;  // buffer cache policy: device scope
constexpr int B3_T = 128;  // tile edge: 128 x 128 outputs, 2 x 2 waves of 64 x 64

__device__ __forceinline__ uint32_t b3_cvt(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, b2));
}
__device__ __forceinline__ float b3_lo(uint32_t p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float b3_hi(uint32_t p) { return __builtin_bit_cast(float, p & 0xFFFF0000u); }

// Two floats (consecutive k of one row) times 2^24 as three packed bf16 pairs.
constexpr float B3_UP = 0x1p24f, B3_DOWN = 0x1p-48f;
__device__ __forceinline__ void b3_split(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
    x *= B3_UP;
    y *= B3_UP;
    h = b3_cvt(x, y);
    const float rx = x - b3_lo(h), ry = y - b3_hi(h);
    m = b3_cvt(rx, ry);
    const uint32_t sx = __builtin_bit_cast(uint32_t, rx - b3_lo(m)), sy = __builtin_bit_cast(uint32_t, ry - b3_hi(m));
    l = __builtin_amdgcn_perm(sy, sx, 0x07060302u);
}

// One operand's slab: 128 rows x 16 G k, 8 floats per thread (256 G threads).
// In LDS each of the three planes holds 16-byte chunks of 8 k of one row, the
// operand a lane of the MFMA takes: chunk (g, plane, half, row) for k = 16 g +
// 8 half + 0..7.
//  - K_CONTIG (nb0 == 4): pieces of four k, 8-byte writes; 4 G lanes cover the
//    64 G contiguous bytes of a row, and the two halves (and groups) of 8 / G
//    rows fill different banks (HS).
//  - R_CONTIG (nb1 == 4): a thread holds four rows at k and k + 1 and writes
//    dwords; rows r mod 4 go to runs of their own (RS apart), so 32 lanes (8
//    rows, 4 pairs of k) write 128 contiguous bytes, and the reads of 8
//    consecutive rows fall on different banks.
//  - GENERIC: K_CONTIG's mapping, element by element.
// Loads go through a buffer resource over the plane: rows past the operand get
// an offset past it (read 0), and k past K is set to 0 where the last slab is
// converted. An R_CONTIG quad that holds the operand's last row may hold up to
// three rows after it, whatever lies there: they reach only sums outside dst.
// 4-byte alignment is enough for the 16-byte loads.
// NP: pieces per thread; 1 leaves rows 64 to 127 out (not R_CONTIG), for a tile whose
// last 64 columns lie past dst.
template <int MODE, int G, int NP = 2>
struct B3Slab {
    static_assert(NP == 2 || MODE != MM_R_CONTIG, "a row-contiguous piece is four rows of one k");
    static constexpr int RS = MODE == MM_R_CONTIG ? 32 * 16 + 32 : 0;
    static constexpr int HS = MODE == MM_R_CONTIG ? 4 * RS : (G == 1 ? 128 * 16 + 128 : 128 * 16 + 64);
    static constexpr int PS = 2 * HS, GS = 3 * PS;
    static constexpr int BYTES = G * GS;
    uint32_t vo[NP];  // byte offset of piece u of slab 0
    int ko[NP];       // its first k within a slab
    uint32_t lo;      // LDS byte offset of piece 0
    uint32_t nb0;
    uint32_t step;    // bytes from one slab to the next
    __amdgpu_buffer_rsrc_t rs;
    f4 r[2][NP];      // [stage][piece]: slab s waits in stage s % 2

    static __device__ __forceinline__ uint32_t chunk(int row) {
        if constexpr (MODE == MM_R_CONTIG) return (uint32_t) ((row & 3) * RS + (row >> 2) * 16);
        else return (uint32_t) row * 16;
    }
    // base: the operand's plane; row0: the tile's first row (the resource begins
    // there, so that only 128 rows have to lie within 32-bit offsets)
    __device__ __forceinline__ void init(const uint8_t* base, int64_t nbk, int64_t nbr, int64_t row0, int64_t nrows,
                                         int64_t K, int64_t k0, int tid) {
        const int rows = nrows - row0 < B3_T ? (int) (nrows - row0) : B3_T;
        rs = __builtin_amdgcn_make_buffer_rsrc((void*) (base + row0 * nbr), (short) 0,
                                               (int) ((rows - 1) * nbr + (K - 1) * nbk + 4), MM_RSRC_WORD3);
        nb0 = (uint32_t) nbk;
        step = (uint32_t) (16 * G * nbk);
        if constexpr (MODE == MM_R_CONTIG) {
            const int lane = tid & 63, wave = tid >> 6;
            const int q = 8 * (wave & 3) + (lane & 7), kp = (lane >> 3) & 7, g = wave >> 2;
#pragma unroll
            for (int u = 0; u < NP; ++u) {
                ko[u] = 16 * g + 2 * kp + u;
                vo[u] = 4 * q < rows ? (uint32_t) ((k0 + ko[u]) * nbk + 16 * q) : MM_OUT;
            }
            lo = (uint32_t) (g * GS + (kp >> 2) * HS + q * 16 + (kp & 3) * 4);
        } else {
            const int row = tid / (4 * G), kq = tid % (4 * G);
#pragma unroll
            for (int u = 0; u < NP; ++u) {
                ko[u] = 4 * kq;
                vo[u] = row + 64 * u < rows ? (uint32_t) ((row + 64 * u) * nbr + (k0 + ko[u]) * nbk) : MM_OUT;
            }
            lo = (uint32_t) ((kq >> 2) * GS + ((kq >> 1) & 1) * HS + row * 16 + (kq & 1) * 8);
        }
    }
    // piece u of slab s (0 past the part's n slabs)
    __device__ __forceinline__ f4 fetch(int s, int n, int u) const {
        const uint32_t so = s < n ? (uint32_t) s * step : MM_PAST;
        f4 v;
        if constexpr (MODE == MM_GENERIC) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                     rs, vo[u] == MM_OUT ? MM_OUT : vo[u] + e * nb0, so, 0));
        } else {
            v = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo[u], so, 0));
        }
        return v;
    }
    __device__ __forceinline__ void load(int st, int s, int n, int u) { r[st][u] = fetch(s, n, u); }
    // k past K of the last slab, whose first k is `left` before K, becomes 0
    __device__ __forceinline__ void mask(int st, int left) {
#pragma unroll
        for (int u = 0; u < NP; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ko[u] + (MODE == MM_R_CONTIG ? 0 : e) >= left) r[st][u][e] = 0.f;
    }
    // half u of the registers, split, into the planes at l: piece u, or
    // (R_CONTIG) rows 2u and 2u + 1 of the four, whose k pair is in both pieces
    __device__ __forceinline__ void store(int st, uint8_t* l, int u) const {
        if constexpr (MODE == MM_R_CONTIG) {
#pragma unroll
            for (int j = 2 * u; j < 2 * u + 2; ++j) {
                uint32_t h, m, t;
                b3_split(r[st][0][j], r[st][1][j], h, m, t);
                uint8_t* d = l + lo + j * RS;
                *(uint32_t*) d = h;
                *(uint32_t*) (d + PS) = m;
                *(uint32_t*) (d + 2 * PS) = t;
            }
        } else {
            u2 h, m, t;
            uint32_t a, b, c;
            b3_split(r[st][u].x, r[st][u].y, a, b, c);
            h.x = a, m.x = b, t.x = c;
            b3_split(r[st][u].z, r[st][u].w, a, b, c);
            h.y = a, m.y = b, t.y = c;
            uint8_t* d = l + lo + u * 64 * 16;
            *(u2*) d = h;
            *(u2*) (d + PS) = m;
            *(u2*) (d + 2 * PS) = t;
        }
    }
    // as floats [k][row] for the FP32 instructions
    static constexpr int LDF = B3_T + 1;
    __device__ __forceinline__ void store_f32(float* l, int tid) const {
#pragma unroll
        for (int u = 0; u < NP; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (MODE == MM_R_CONTIG) {
                    const int q = 8 * ((tid >> 6) & 3) + (tid & 7);
                    l[ko[u] * LDF + 4 * q + e] = r[0][u][e];
                } else {
                    l[(ko[u] + e) * LDF + tid / (4 * G) + 64 * u] = r[0][u][e];
                }
            }
    }
    static __device__ __forceinline__ b8 frag(const uint8_t* l, int plane, uint32_t at) {
        return __builtin_bit_cast(b8, *(const u4*) (l + at + plane * PS));
    }
};

template <int AMODE, int BMODE, int G>
constexpr int b3_lds() {
    return 3 * (B3Slab<AMODE, G>::BYTES + B3Slab<BMODE, G>::BYTES);
}

// Where a workgroup's tile lies: its operands' planes, its dst plane, its first row
// and column, its number and its part of K (all uniform).
struct B3Place {
    const uint8_t* a;
    const uint8_t* b;
    uint8_t* d;
    int64_t i0, j0;
    uint32_t tile;
    int part;
};

// One 128 x 128 tile (of one part of K) on G groups of 4 waves;
// group g multiplies k = 16 g .. 16 g + 15 of every 16 G deep slab, and with two
// groups their sums meet in LDS at the end. Three slab buffers take turns:
// during the MFMAs of slab s, whose operands are in registers, those of slab s +
// 1 are read from the second buffer, slab s + 2 is split and stored into the
// third, and slab s + 4 is loaded into the registers that held s + 2; one
// barrier per slab.
// NY: 32-column blocks per wave, 1 where the tile's last 64 columns lie past dst.
template <int AMODE, int BMODE, int G, int MEET, bool ACC, int NY>
__device__ __forceinline__ void b3_tile(const MMArgs& p, const B3Place& at, uint8_t* lds) {
    static_assert(!ACC || MEET == B3_ALONE, "parts that meet store or add to a dst of their own");
    using SA = B3Slab<AMODE, G>;
    constexpr int NPB = NY == 1 && BMODE != MM_R_CONTIG ? 1 : 2;
    using SB = B3Slab<BMODE, G, NPB>;
    constexpr int BK = 16 * G;
    constexpr int BUF = SA::BYTES + SB::BYTES;
    constexpr int RED = G == 2 ? 4 * 64 * 64 * 4 : 0;  // half of every wave's sums
    constexpr int F32 = 2 * BK * SA::LDF * 4;
    static_assert(RED <= 3 * BUF && F32 <= 3 * BUF, "the slab buffers hold what comes after them");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wi = wave & 1, wj = (wave >> 1) & 1, grp = wave >> 2;
    const int half = lane >> 5, col = lane & 31;

    const int64_t i0 = at.i0, j0 = at.j0;
    const int part = at.part;
    const uint32_t tile = at.tile;
    uint8_t* d = at.d;
    const int slabs = (int) ((p.K + BK - 1) / BK);
    const int per_part = (slabs + (int) p.parts - 1) / (int) p.parts;
    const int kt0 = part * per_part;
    const int nk = slabs - kt0 < per_part ? slabs - kt0 : per_part;
    // k left from the part's last slab on (BK and more: the slab is whole)
    const int64_t left64 = p.K - (int64_t) (kt0 + nk - 1) * BK;
    const int left = left64 > BK ? BK : (int) left64;

    SA sa;
    SB sb;
    sa.init(at.a, p.a_nb0, p.a_nb1, i0, p.M, p.K, (int64_t) kt0 * BK, tid);
    sb.init(at.b, p.b_nb0, p.b_nb1, j0, p.N, p.K, (int64_t) kt0 * BK, tid);

    // the products of first parts, and the smaller ones: a bf16 instruction drops
    // what lies below its accumulator's last bit, downwards, which the small
    // products added to the large sums would suffer from (2-norm 0.99e-6 instead of
    // 0.40e-6 at K = 4096, and a mean of -1.8e-7 of the result's)
    f16v acc[2][NY], cor[2][NY];
    auto clear = [&]() {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[x][y][v] = 0.f;
    };
    auto gload = [&](int st, int kt) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            sa.load(st, kt, nk, u);
            if (u < NPB) sb.load(st, kt, nk, u);
        }
    };
    auto lstore = [&](int st, uint8_t* l) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            sa.store(st, l, u);
            if (u < NPB) sb.store(st, l + SA::BYTES, u);
        }
    };
    auto masked = [&](int st, int kt) {
        if (kt == nk - 1 && left < BK) {
            sa.mask(st, left);
            sb.mask(st, left);
        }
    };
    // slabs 0 to 3 are all asked for at once: the first two wait here, the next
    // two in the registers' two stages
    gload(0, 0);
    gload(1, 1);
    f4 ahead[2][2][2];
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ahead[st][0][u] = sa.fetch(2 + st, nk, u);
            if (u < NPB) ahead[st][1][u] = sb.fetch(2 + st, nk, u);
        }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        masked(st, st);
        lstore(st, lds + st * BUF);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            sa.r[st][u] = ahead[st][0][u];
            if (u < NPB) sb.r[st][u] = ahead[st][1][u];
        }
    }
    __syncthreads();

    uint32_t ao[2], bo[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        ao[x] = grp * SA::GS + half * SA::HS + SA::chunk(wi * 64 + x * 32 + col);
        bo[x] = SA::BYTES + grp * SB::GS + half * SB::HS + SB::chunk(x * 64 + wj * 32 + col);
    }
    clear();
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) cor[x][y] = acc[x][y];
    // The operands of a slab are replaced by the next slab's as soon as a
    // product is the last to use them; the order of the products leaves four
    // MFMAs between each such read and the first use of what it reads.
    b8 fa[3][2], fb[3][2];
    auto fragsA = [&](const uint8_t* l, int pl) {
#pragma unroll
        for (int x = 0; x < 2; ++x) fa[pl][x] = SA::frag(l, pl, ao[x]);
    };
    auto fragsB = [&](const uint8_t* l, int pl) {
#pragma unroll
        for (int y = 0; y < NY; ++y) fb[pl][y] = SB::frag(l, pl, bo[y]);
    };
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
        fragsA(lds, pl);
        fragsB(lds, pl);
    }
    int b1 = BUF, b2 = 2 * BUF;  // LDS offsets of slabs kt + 1 and kt + 2
    // (a slab past the part's last, where their number is odd, is one of zeros)
    auto slab = [&](int kt, auto parity, auto last) {
        constexpr int ST = decltype(parity)::value;
        const uint8_t* rd = lds + b1;
        uint8_t* nxt = lds + b2;
        if constexpr (decltype(last)::value) masked(ST, kt + 2);
        // m m, l h, h l, m h, h m into the small sums, h h into the large ones
        constexpr int PA[6] = {1, 2, 0, 1, 0, 0}, PB[6] = {1, 0, 2, 0, 1, 0};
#pragma unroll
        for (int q = 0; q < 6; ++q) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < NY; ++y) {
                    f16v& c = q < 5 ? cor[x][y] : acc[x][y];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[PB[q]][y], fa[PA[q]][x], c, 0, 0, 0);
                }
            if (q == 1) fragsA(rd, 2), sa.store(ST, nxt, 0);
            if (q == 2) fragsB(rd, 2), sa.store(ST, nxt, 1);
            if (q == 3) fragsA(rd, 1), sb.store(ST, nxt + SA::BYTES, 0);
            if (q == 4) fragsB(rd, 1);
            if (q == 4 && NPB == 2) sb.store(ST, nxt + SA::BYTES, NPB - 1);
            if (q == 5) fragsA(rd, 0), fragsB(rd, 0);
            if constexpr (!decltype(last)::value) {
                if (q == 2) sa.load(ST, kt + 4, nk, 0), sa.load(ST, kt + 4, nk, 1);
                if (q == 4) sb.load(ST, kt + 4, nk, 0);
                if (q == 4 && NPB == 2) sb.load(ST, kt + 4, nk, NPB - 1);
            }
            // after each MFMA at most two LDS accesses, a load and six vector
            // instructions (left to itself the compiler moves the conversion
            // ahead of the MFMAs: forward product 103.6 -> 91.9 us)
#pragma unroll
            for (int z = 0; z < 2 * NY; ++z) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x300, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
        }
        const int b0 = 3 * BUF - b1 - b2;
        b1 = b2;
        b2 = b0;
        __syncthreads();
    };
    using zero = std::integral_constant<int, 0>;
    using one = std::integral_constant<int, 1>;
    int kt = 0;
    for (; kt + 4 < nk; kt += 2) {
        slab(kt, zero{}, std::false_type{});
        slab(kt + 1, one{}, std::false_type{});
    }
    // at most four slabs are left: the last is among those stored here, and what
    // would be loaded nobody multiplies
    for (; kt < nk; kt += 2) {
        slab(kt, zero{}, std::true_type{});
        slab(kt + 1, one{}, std::true_type{});
    }

    // accumulator register v of tile (x, y) holds the tile's dst row i = ib + 32 x +
    // col and column j = jb + 64 y + 8 (v / 4) + 4 half + v % 4
    const int ib = wi * 64, jb = wj * 32;
    const int rows = p.M - i0 < B3_T ? (int) (p.M - i0) : B3_T, cols = p.N - j0 < B3_T ? (int) (p.N - j0) : B3_T;
    // a result that is not finite: the same sums on the FP32 instructions. Sums
    // outside dst don't count (they can hold rows that are not the operand's).
    float most = 0.f;  // of the results' magnitudes, NaN where one is
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        float mx = 0.f;
#pragma unroll
        for (int y = 0; y < NY; ++y) {
            const int rest = cols - (jb + y * 64 + 4 * half);
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[x][y][v] = (acc[x][y][v] + cor[x][y][v]) * B3_DOWN;
                if (cols == B3_T || 8 * (v >> 2) + (v & 3) < rest)
                    mx = __builtin_elementwise_maximum(mx, __builtin_fabsf(acc[x][y][v]));
            }
        }
        if (ib + x * 32 + col < rows) most = __builtin_elementwise_maximum(most, mx);
    }
    if (__syncthreads_or(!(most < __builtin_inff()))) {
        clear();
        float* la = (float*) lds;
        float* lb = la + BK * SA::LDF;
        for (int k0 = 0; k0 < nk; ++k0) {
            gload(0, k0);
            masked(0, k0);
            sa.store_f32(la, tid);
            sb.store_f32(lb, tid);
            __syncthreads();
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int k = 16 * grp + 2 * s + half;
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < NY; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(lb[k * SA::LDF + y * 64 + wj * 32 + col],
                                                                         la[k * SA::LDF + wi * 64 + x * 32 + col],
                                                                         acc[x][y], 0, 0, 0);
            }
            __syncthreads();
        }
    }

    constexpr int NX = G == 2 ? 1 : 2;
    int x0 = 0;
    if constexpr (G == 2) {
        // each group gives the other the sums of one x and keeps its own x = grp
        float* red = (float*) lds + (wave & 3) * 64 * 64 + lane;
        float* mine = red;
        // lds is idle: the last slab and the repeated sums end with a barrier
        if (grp == 1) {
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int v = 0; v < 16; ++v) mine[(y * 16 + v) * 64] = acc[0][y][v];
        } else {
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int v = 0; v < 16; ++v) mine[(32 + y * 16 + v) * 64] = acc[1][y][v];
        }
        __syncthreads();
        x0 = grp;
        if (grp == 0) {
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[0][y][v] += red[(y * 16 + v) * 64];
        } else {
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[0][y][v] = red[(32 + y * 16 + v) * 64] + acc[1][y][v];
        }
    }
    d += i0 * p.d_nb0 + j0 * p.d_nb1;
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(
        (void*) d, (short) 0, (int) ((rows - 1) * p.d_nb0 + (cols - 1) * p.d_nb1 + 4), MM_RSRC_WORD3);
    const uint32_t nb1 = (uint32_t) p.d_nb1;
    uint32_t* tk = MEET != B3_ALONE ? p.tickets + 2 * (tile * 4 * G + wave) : nullptr;
    bool second = false;
    if constexpr (MEET == B3_PAIR) {
        second = !ticket_first(tk, lane);
        if (second) ticket_wait(tk, lane);
    }
    if constexpr (MEET == B3_SLOTS) {
        // every part's 16 NX y blocks of a wave are stored as float4s of a lane,
        // written through to where every XCD reads them (sc1); the part that
        // takes the last ticket adds them up in part order and goes on to dst
        constexpr int W = 4 * G * NX * 8;  // float4 x 64 lanes of all waves of a slot (64 KiB)
        constexpr int NB = NX * NY * 4;
        auto slot = [&](int q) {
            return __builtin_amdgcn_make_buffer_rsrc((void*) (p.slots + ((int64_t) tile * p.parts + q) * W * 256),
                                                     (short) 0, W * 1024, MM_RSRC_WORD3);
        };
        const uint32_t wo = (uint32_t) (wave * NX * 8 * 1024 + lane * 16);
        if (!ticket_last(tk, lane, p.parts)) {
            const __amdgpu_buffer_rsrc_t rq = slot(part);
#pragma unroll
            for (int x = 0; x < NX; ++x)
#pragma unroll
                for (int y = 0; y < NY; ++y)
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const f4 v = {acc[x][y][4 * c], acc[x][y][4 * c + 1], acc[x][y][4 * c + 2], acc[x][y][4 * c + 3]};
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), rq, wo,
                                                               ((x * NY + y) * 4 + c) * 1024, B3_SC1);
                    }
            ticket_arrive(tk, lane);
            return;
        }
        ticket_wait_all(tk, lane, p.parts - 1);
        f4 sum[NB];
        for (int q = 0; q < (int) p.parts; ++q) {
            const __amdgpu_buffer_rsrc_t rq = slot(q);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                f4 v;
                if (q == part) {
                    const f16v& s = acc[b / (4 * NY)][(b >> 2) % NY];
                    const int c = 4 * (b & 3);
                    v = (f4){s[c], s[c + 1], s[c + 2], s[c + 3]};
                } else {
                    v = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rq, wo, b * 1024, B3_SC1));
                }
                sum[b] = q == 0 ? v : sum[b] + v;
            }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[b / (4 * NY)][(b >> 2) % NY][4 * (b & 3) + c] = sum[b][c];
        ticket_clear(tk, lane);
    }
#pragma unroll
    for (int x = 0; x < NX; ++x) {
        const int i = ib + (x0 + x) * 32 + col;
#pragma unroll
        for (int y = 0; y < NY; ++y) {
            const int j = jb + y * 64 + 4 * half;
            const uint32_t vo = i < rows ? (uint32_t) (i * p.d_nb0 + j * p.d_nb1) : MM_OUT;
            const int rest = cols - j;  // columns from j on
            auto off = [&](int v) { return cols == B3_T || 8 * (v >> 2) + (v & 3) < rest ? vo : MM_OUT; };
            auto so = [&](int v) { return (uint32_t) (8 * (v >> 2) + (v & 3)) * nb1; };
            if constexpr (MEET == B3_PAIR) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    if (off(v) == MM_OUT) continue;
                    float* o = (float*) (d + vo + so(v));
                    if (second) __hip_atomic_fetch_add(o, acc[x][y][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else __hip_atomic_store(o, acc[x][y][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            } else if constexpr (ACC) {
                float old[16];
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    old[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, off(v), so(v), 0));
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, old[v] + acc[x][y][v]), rd,
                                                          off(v), so(v), 0);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                // aux 2 (nt): dst is not read again by this launch
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float o = acc[x][y][v];  // (a bit_cast of a vector's element would read element 0)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o), rd, off(v), so(v), 2);
                }
            }
        }
    }
    if constexpr (MEET == B3_PAIR) {
        if (second) ticket_clear(tk, lane);
        else ticket_publish(tk, lane);
    }
}

template <int AMODE, int BMODE, int G, int MEET, bool ACC, bool NARROW>
__global__ __launch_bounds__(256 * G, 2) void k_mm_bf3(MMArgs p) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[b3_lds<AMODE, BMODE, G>()];
    // 32-bit divisions: the grid is under 2^31
    uint32_t t = blockIdx.x;
    const uint32_t tiles_i = (uint32_t) p.tiles_i, tiles_j = (uint32_t) p.tiles_j;
    if (p.xcd_planes) {
        const uint32_t tpp = tiles_i * tiles_j * (MEET == B3_ALONE ? 1 : p.parts), x = t & 7, k = t >> 3;
        t = (8 * (k / tpp) + x) * tpp + k % tpp;
    }
    uint32_t part_ = (uint32_t) p.part;
    if constexpr (MEET != B3_ALONE) {
        part_ = t % p.parts;
        t /= p.parts;
    }
    // the divisions run on the vector unit: back to scalars, so that addresses and
    // buffer resources are too
    const int part = (int) __builtin_amdgcn_readfirstlane(part_);
    const uint32_t tile = __builtin_amdgcn_readfirstlane(t);
    const uint32_t ti = __builtin_amdgcn_readfirstlane(tile % tiles_i);
    const uint32_t tt = __builtin_amdgcn_readfirstlane(tile / tiles_i);
    const uint32_t tj = __builtin_amdgcn_readfirstlane(tt % tiles_j);
    const uint32_t plane = __builtin_amdgcn_readfirstlane(tt / tiles_j);
    const uint32_t i2 = __builtin_amdgcn_readfirstlane(plane % (uint32_t) p.b_ne2);
    const uint32_t i3 = __builtin_amdgcn_readfirstlane(plane / (uint32_t) p.b_ne2);
    const uint32_t a2 = __builtin_amdgcn_readfirstlane(i2 % (uint32_t) p.a_ne2);
    const uint32_t a3 = __builtin_amdgcn_readfirstlane(i3 % (uint32_t) p.a_ne3);
    B3Place at;
    at.a = p.a + (int64_t) a2 * p.a_nb2 + (int64_t) a3 * p.a_nb3;
    at.b = p.b + (int64_t) i2 * p.b_nb2 + (int64_t) i3 * p.b_nb3;
    at.d = p.d + (int64_t) i2 * p.d_nb2 + (int64_t) i3 * p.d_nb3;
    at.i0 = (int64_t) ti * B3_T;
    at.j0 = (int64_t) tj * B3_T;
    at.tile = tile;
    at.part = part;
    // NARROW: the last column of tiles is (elsewhere that copy of the tile is left out)
    if (NARROW && p.N - at.j0 <= 64) b3_tile<AMODE, BMODE, G, MEET, ACC, 1>(p, at, lds);
    else b3_tile<AMODE, BMODE, G, MEET, ACC, 2>(p, at, lds);
}

int mode_of(int64_t nb0, int64_t nb1) {
    return nb0 == 4 ? MM_K_CONTIG : nb1 == 4 ? MM_R_CONTIG : MM_GENERIC;
}

template <int G, int MEET, bool ACC>
int b3_launch(const MMArgs& p, unsigned grid, hipStream_t s) {
    int am = mode_of(p.a_nb0, p.a_nb1), bm = mode_of(p.b_nb0, p.b_nb1);
    const bool narrow = (p.N - 1) % B3_T < 64;
#define TRC_B3(A, B) \
    if (am == A && bm == B) {                                                                              \
        if (narrow) hipLaunchKernelGGL((k_mm_bf3<A, B, G, MEET, ACC, true>), dim3(grid), dim3(256 * G), 0, s, p); \
        else hipLaunchKernelGGL((k_mm_bf3<A, B, G, MEET, ACC, false>), dim3(grid), dim3(256 * G), 0, s, p);       \
    }
    // an operand that runs along neither dimension is rare: both load by element
    if (am == MM_GENERIC || bm == MM_GENERIC) am = bm = MM_GENERIC;
    TRC_B3(MM_K_CONTIG, MM_K_CONTIG)
    TRC_B3(MM_K_CONTIG, MM_R_CONTIG)
    TRC_B3(MM_R_CONTIG, MM_K_CONTIG)
    TRC_B3(MM_R_CONTIG, MM_R_CONTIG)
    TRC_B3(MM_GENERIC, MM_GENERIC)
#undef TRC_B3
    return check_launch("mul_mat_f32 (three bf16)");
}

}  // namespace
}  // namespace trc_hip
