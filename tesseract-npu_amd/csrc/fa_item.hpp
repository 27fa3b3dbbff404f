// fa_item.hpp -- the work items of FLASH_ATTN_EXT, shared by the host planner (fa_plan.hpp) and the kernels.
#pragma once

#include <stdint.h>

namespace tsr {

// One chunk of one query token (the planner's output), in execution order per token.
struct FaItem {
    uint32_t t;              // token
    uint32_t u0, n;          // groups [u0, u0 + n)
    uint32_t c_lo, c_hi;     // visible chunk-relative cells (FAST)
    uint32_t general;        // GENERAL chunk: all cells, f32 mask added
    uint32_t s_off;          // first score cell of the item in S (scores at S + s_off * n_head)
    uint32_t tile0, ntiles;  // its 256-cell score tiles (rows tile0 .. tile0 + ntiles - 1 of Mpart)
};
// The P.V segments (4 of a channel's groups, which are every fourth one of the item's) of an item of that many groups:
// the most of its four channels. The planner cuts items at 128 groups.
constexpr uint32_t kMaxSegments = 8;
constexpr uint32_t fa_segments(uint32_t groups) { return groups > 16u ? (groups + 15u) / 16u : 1u; }
constexpr uint32_t kFaInlItems = 48, kFaInlTok = 8;   // the largest work list that travels in the kernel arguments

}  // namespace tsr
