// The bf16 tile kernel (mm_bf3.h) with K whole, and the choice and launch of its
// tiles. The parts of K that meet are in mm_bf3_parts.hip.
#include "mm_bf3.h"

namespace trc_hip {

int launch_mm_bf3_pair(const MMArgs& p, unsigned grid, hipStream_t s);
int launch_mm_bf3_slots(const MMArgs& p, unsigned grid, hipStream_t s);

bool mm_bf3_fits(const MMArgs& p) {
    // 32-bit buffer offsets over the rows of a tile, those included that are formed
    // for what is not there: k up to the end of its slab, and the columns of a wave's
    // 32 x 32 block, the last 27 after the one its lanes' offsets name
    auto span = [](int64_t n0, int64_t nb0, int64_t n1, int64_t nb1) { return (n0 - 1) * nb0 + (n1 - 1) * nb1 + 4; };
    const int64_t k = (p.K + 31) / 32 * 32;
    const int64_t ti = p.M < B3_T ? p.M : B3_T, tj = p.N < B3_T ? p.N : B3_T;
    return span(k, p.a_nb0, ti, p.a_nb1) <= MM_PAST && span(k, p.b_nb0, tj, p.b_nb1) <= MM_PAST &&
           span(ti, p.d_nb0, tj < 28 ? 28 : tj, p.d_nb1) <= MM_PAST;
}

B3Plan mm_bf3_plan(const MMArgs& p, int64_t planes, int max_parts) {
    // Times in us, measured where one workgroup of 8 waves has a CU: a 32-deep
    // slab 0.8, a launch with K whole 7.5 (6.4 to 9, K = 130 to 4096), with K in parts 8 +
    // 1.6 per part (16 to 64 tiles; two parts that meet in dst 12, six 17, eight
    // 19 to 24). 4096 x 4096 x 128, parts 1, 2, 3, 4, 6, 8: 107.6, 63.0, 45.5,
    // 38.9, 34.9, 39.2; 1024 x 1024 x 512: 32.3, 25.1, 20.6, 20.9, 21.9, 27.2.
    // Operands that run along neither dimension load element by element, and with
    // them the other operand: a slab takes 2.4 with one such operand, 3.3 with two
    // (0.6 of that with up to 64 columns; with up to 64 rows 0.65, or 0.35), and a
    // launch that fills the chip 12 more, 6 with up to 64 columns (256 x 256 x 512 in
    // two parts 35 and 42, 1408 x 1408 x 1024 60 and 74, 1408 x 1408 x 512 40 and 47). K
    // whole, two workgroups to a CU and src0 strided 3.5 for each tile of a CU (4096 x
    // 4096 x 512 231, with src1 strided 150).
    const int64_t tiles = ((p.M + B3_T - 1) / B3_T) * ((p.N + B3_T - 1) / B3_T) * planes;
    const int64_t cus = device_cus();
    const double slabs = (double) ((p.K + 31) / 32);
    const bool sa = mm_a_strided(p), sb = mm_b_strided(p);
    const bool narrow = p.N <= 64, strided = sa || sb;
    const double part_of = p.M <= 64 ? (narrow ? 0.35 : 0.65) : narrow ? 0.6 : 1;
    const double slab = strided ? (sa && sb ? 3.3 : 2.4) * part_of : narrow ? 0.7 : 0.8;
    const double slab1 = sa && !sb && tiles > cus ? 3.5 * part_of : slab;
    auto base = [&](int64_t groups) {
        return strided ? (narrow ? 6 : 12) * (groups < cus ? (double) groups / cus : 1.0) : 0;
    };
    const double rounds = strided && tiles > cus ? (double) tiles / cus : (double) ((tiles + cus - 1) / cus);
    B3Plan best{2, 1, base(tiles) + 7.5 + slab1 * slabs * rounds};
    for (int parts = 2; parts <= max_parts; ++parts) {
        // a part is at least 4 slabs: shorter ones are all launch and meeting
        if (slabs < 4 * parts || tiles * parts > (parts == 2 ? 4 * cus : cus)) break;
        if (parts > 2 && tiles * parts > (int64_t) MM_SLOTS) break;
        if (tiles * 16 > MM_TICKETS) break;
        const double each = (double) (((int64_t) slabs + parts - 1) / parts);
        const double us = base(tiles * parts) + 8 + 1.6 * parts + slab * each * (double) ((tiles * parts + cus - 1) / cus);
        if (us < best.us) best = {2, parts, us};
    }
    // More tiles than CUs with K whole: 4-wave workgroups, two to a CU, whose
    // prologues and stores overlap the other's MFMAs (4096 x 4096 x 512 99 ->
    // 90 us, configuration 4 143 -> 106 us).
    if (best.parts == 1 && tiles > cus) best.groups = 1;
    return best;
}

int launch_mm_bf3(MMArgs& p, int64_t planes, int groups, int parts, bool acc, hipStream_t s) {
    p.tiles_i = (p.M + B3_T - 1) / B3_T;
    p.tiles_j = (p.N + B3_T - 1) / B3_T;
    p.xcd_planes = planes % 8 == 0 ? 1 : 0;
    const int64_t tiles = p.tiles_i * p.tiles_j * planes;
    if (tiles * parts > max_groups(256 * groups)) {
        return fail(TRC_HIP_E_SHAPE, "mul_mat: %lld workgroups exceed one launch", (long long) tiles * parts);
    }
    const unsigned n = (unsigned) tiles;
    // parts of whole slabs, none of them empty
    const int64_t slabs = (p.K + 16 * groups - 1) / (16 * groups), per = (slabs + parts - 1) / parts;
    p.parts = (uint32_t) ((slabs + per - 1) / per);
    p.part = 0;
    if (p.parts > 1) {
        float* slots = nullptr;
        const bool pair = p.parts == 2;
        const int rc = mm_stream_scratch(s, pair ? 0 : (size_t) tiles * p.parts, &p.tickets, &slots);
        if (rc != TRC_HIP_OK) return rc;
        p.slots = slots;
        if (p.tickets != nullptr && pair) return launch_mm_bf3_pair(p, n * 2, s);
        if (p.tickets != nullptr) return launch_mm_bf3_slots(p, n * p.parts, s);
        // no workspace to meet in: one launch after another, each part added to dst
        for (; p.part < (int) p.parts; ++p.part) {
            const int lrc = p.part == 0 ? b3_launch<2, B3_ALONE, false>(p, n, s) : b3_launch<2, B3_ALONE, true>(p, n, s);
            if (lrc != TRC_HIP_OK) return lrc;
        }
        return TRC_HIP_OK;
    }
    if (acc) return groups == 2 ? b3_launch<2, B3_ALONE, true>(p, n, s) : b3_launch<1, B3_ALONE, true>(p, n, s);
    return groups == 2 ? b3_launch<2, B3_ALONE, false>(p, n, s) : b3_launch<1, B3_ALONE, false>(p, n, s);
}

}  // namespace trc_hip
