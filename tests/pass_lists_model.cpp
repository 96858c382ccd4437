// Host model of the lists of an edge-list call (mdet_amd/csrc/pass_lists.h):
// tiles reserve slots and records, the refinement writes the records of the
// tiles that got a slot and fit, readers go by records_written; and passes are
// repeated with grow_lists until everything fits.  Prints what
// tests/test_pass_lists.py checks.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "../mdet_amd/csrc/pass_lists.h"

using namespace mdet;

// One pass over an input whose lists would come out as `full` (cand: the first
// pass's, fb_cand the full rows'), cut by what there is room for: entries past a
// list's end are counted, but not worked on.
static PassCounts pass(const PassCounts& full, uint64_t fb_cand, const PassCaps& cap, bool full_rows) {
    auto share = [](uint64_t whole, uint64_t part, uint64_t of) {
        return part >= of ? whole : (uint64_t)((double)whole * (double)part / (double)of);
    };
    PassCounts n{};
    n.list = full.list;
    n.surv = share(full.surv, cap.list, full.list);
    n.cand = share(full.cand, cap.list, full.list);
    PassCaps unused = cap;
    if (!full_rows || grow_lists(n, unused)) return n;  // the host looks before the full rows
    n.fb_list = full.fb_list;
    n.fb_surv = share(full.fb_surv, cap.fb_list, full.fb_list);
    n.cand += share(fb_cand, cap.fb_list, full.fb_list);
    return n;
}

int main() {
    std::mt19937_64 rng(7);
    auto below = [&](uint64_t n) { return n ? rng() % n : 0; };
    long failed[2] = {0, 0}, most[2] = {0, 0};
    for (int trial = 0; trial < 40000; ++trial) {
        auto length = [&] { return 1 + below(1ull << (1 + below(40))); };
        const bool full_rows = trial & 1;
        const PassCounts full{length(), length(), length(), length(), length()};
        const uint64_t fb_cand = length();
        PassCaps cap{length(), length(), length(), length()};
        int passes = 1;
        while (passes <= PASS_MAX && grow_lists(pass(full, fb_cand, cap, full_rows), cap)) ++passes;
        failed[full_rows] += passes > PASS_MAX;
        most[full_rows] = std::max<long>(most[full_rows], passes);
    }
    long reads = 0, unwritten_read = 0, gaps = 0, refused_whole = 0;
    for (int trial = 0; trial < 20000; ++trial) {
        const uint64_t tiles = 1 + below(60);
        std::vector<uint64_t> count(tiles);
        for (auto& c : count) c = 1 + below(1024);
        uint64_t total = 0;
        for (uint64_t c : count) total += c;
        PassCaps cap{};
        // around the lengths that come out, over and under
        cap.surv = below(2) ? tiles + below(3) : below(tiles + 3);
        cap.cand = below(2) ? total + below(3) : below(total + 600);
        PassCounts n{};
        std::vector<char> written(cap.cand, 0);
        // two passes share the survivor list (first pass, then the full rows' own slots)
        const uint64_t split = below(3) ? tiles : below(tiles + 1);
        for (uint64_t t = 0; t < tiles; ++t) {
            uint64_t& cnt = t < split ? n.surv : n.fb_surv;
            const uint64_t slot = cnt++, base = n.cand;
            n.cand += count[t];
            if (slot >= cap.surv || base + count[t] > cap.cand) continue;
            for (uint64_t k = 0; k < count[t]; ++k) written[base + k] = 1;
        }
        bool whole = n.cand <= cap.cand;
        for (uint64_t k = 0; k < n.cand && k < cap.cand; ++k) whole = whole && written[k];
        gaps += !whole;
        if (records_written(n, cap)) {
            ++reads;
            unwritten_read += !whole;
        } else {
            refused_whole += whole;
        }
    }
    std::printf("failed %ld failed_full_rows %ld most %ld most_full_rows %ld limit %d\n", failed[0], failed[1], most[0],
                most[1], PASS_MAX);
    std::printf("reads %ld unwritten_read %ld gaps %ld refused_whole %ld\n", reads, unwritten_read, gaps, refused_whole);
    return 0;
}
