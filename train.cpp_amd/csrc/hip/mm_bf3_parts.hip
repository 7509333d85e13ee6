// The bf16 tile kernel (mm_bf3.h) with K in parts that meet in dst or in slots.
#include "mm_bf3.h"

namespace trc_hip {

int launch_mm_bf3_pair(const MMArgs& p, unsigned grid, hipStream_t s) {
    return b3_launch<2, B3_PAIR, false>(p, grid, s);
}

int launch_mm_bf3_slots(const MMArgs& p, unsigned grid, hipStream_t s) {
    return b3_launch<2, B3_SLOTS, false>(p, grid, s);
}

}  // namespace trc_hip
