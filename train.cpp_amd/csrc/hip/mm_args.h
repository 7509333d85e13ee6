// What the F32 mul_mat kernels (mul_mat.hip, mm_bf3.hip) are given.
#pragma once

#include "common.h"

namespace trc_hip {

// How an operand's slabs are loaded: along k (nb0 == 4), along rows (nb1 == 4) or
// element by element.
enum MMLoad { MM_K_CONTIG = 0, MM_R_CONTIG = 1, MM_GENERIC = 2 };

struct MMArgs {
    const uint8_t* a;
    const uint8_t* b;
    uint8_t* d;
    int64_t K, M, N;
    int64_t a_nb0, a_nb1, a_nb2, a_nb3, a_ne2, a_ne3;
    int64_t b_nb0, b_nb1, b_nb2, b_nb3, b_ne2;
    int64_t d_nb0, d_nb1, d_nb2, d_nb3;
    int64_t tiles_i, tiles_j;
    int xcd_planes;  // 1: planes % 8 == 0, tiles of plane p on XCD p % 8
    int64_t d_span;  // bytes from a dst plane's first element to past its last
    uint32_t* tickets;  // K in parts: two words per wave of every tile, zero between launches
    float* slots;       // the parts' sums, 64 KiB per tile and part
    uint32_t parts;     // parts of K
    int part;           // the part of a launch that computes one of them
};

// operands that run along neither dimension: both kernels load these by element
inline bool mm_a_strided(const MMArgs& p) { return p.a_nb0 != 4 && p.a_nb1 != 4; }
inline bool mm_b_strided(const MMArgs& p) { return p.b_nb0 != 4 && p.b_nb1 != 4; }

constexpr uint32_t MM_RSRC_WORD3 = 0x00020000u;  // gfx9 buffer resource: raw 32-bit dwords
constexpr uint32_t MM_OUT = 0x80000000u;         // an offset past the resource: loads read 0, stores drop

// a scalar offset past a plane of at most this many bytes, which MM_OUT can be
// added to without wrapping
constexpr uint32_t MM_PAST = 0x7FFFF000u;

// The bf16 tile kernel (mm_bf3.hip): 128 x 128 tiles on `groups` x 4 waves, K in
// up to `parts` parts (more than one takes 2 groups).
struct B3Plan {
    int groups, parts;
    double us;  // the model's time, to weigh against the FP32 tiles
};
bool mm_bf3_fits(const MMArgs& p);
B3Plan mm_bf3_plan(const MMArgs& p, int64_t planes, int max_parts);
int launch_mm_bf3(MMArgs& p, int64_t planes, int groups, int parts, bool acc, hipStream_t s);

}  // namespace trc_hip
