// Host checks of the rate-control code that the host library and the GPU share
// (libgail_amd/csrc/rc_shared.h). Test infrastructure.
#include "rc_shared.h"

using namespace gail_amd;

extern "C" {

// rc_block_hull_to copies kGroup passes at a time: how many of the entries it copies
// RcPassRows::load leaves unset, for a block of np passes.
int rc_pass_entries_unset(int np) {
    const uint32_t mark = 0xDEADBEEFu;
    uint32_t len[kMaxPasses] = {};
    int32_t dist[kMaxPasses] = {};
    const RcPassRows rows{len, dist};
    constexpr int G = RcPassRows::kGroup;
    int unset = 0;
    for (int k = 0; k < np + G; k += G) {  // as the hull reads: one group ahead
        uint32_t l[4] = {mark, mark, mark, mark};
        int32_t d[4] = {(int32_t)mark, (int32_t)mark, (int32_t)mark, (int32_t)mark};
        rows.load(k, np, l, d);
        if (k >= np) continue;  // not copied
        for (int j = 0; j < G; ++j) unset += (l[j] == mark) + (d[j] == (int32_t)mark);
    }
    return unset;
}

}  // extern "C"
