// The lists of an edge-list call whose lengths only the device finds out
// (tnf_pairs.hip): how long they came out, what was there to hold them, and
// what may be read when one did not fit.  constexpr functions, for the kernels
// and the host alike.
#pragma once

#include <cstdint>

namespace mdet {

// Lengths as the kernels count them, past the capacities too.
struct PassCounts {
    uint64_t list;     // listed tiles
    uint64_t surv;     // tiles with survivors
    uint64_t fb_list;  // the same of the learned filter's full rows
    uint64_t fb_surv;
    uint64_t cand;     // candidate records reserved, by both
};

struct PassCaps {
    uint64_t list, surv, fb_list, cand;  // surv holds either pass's tiles
};

// Whether every reserved candidate record was written.  A tile reserves its
// records together with its slot, so one whose slot lies past the survivor
// list, or whose records reach past the candidates' end, leaves a gap below
// the counted length, which holds whatever the memory held: a record of the
// context's last input or of nobody.  Records are indices into the rows; none
// may be read while this is false.  (Listed tiles that did not fit reserve
// nothing.)
constexpr bool records_written(const PassCounts& n, const PassCaps& cap) {
    return n.surv <= cap.surv && n.fb_surv <= cap.surv && n.cand <= cap.cand;
}

// Raises the capacities that were too small, with some headroom; true if any
// was: the pass has to run again.
constexpr bool grow_lists(const PassCounts& n, PassCaps& cap) {
    bool grown = false;
    auto fit = [&](uint64_t need, uint64_t& c) {
        if (need > c) c = need + need / 4 + 64, grown = true;
    };
    fit(n.list, cap.list);
    fit(n.surv > n.fb_surv ? n.surv : n.fb_surv, cap.surv);
    fit(n.fb_list, cap.fb_list);
    fit(n.cand, cap.cand);
    return grown;
}

// Passes of one call at most.  A list's true length shows only in a pass in
// which the list before it fits: listed tiles, then survivors and candidates,
// then the full rows' listed tiles, then theirs (with all candidates), and the
// pass after that holds everything.
constexpr int PASS_MAX = 5;

}  // namespace mdet
