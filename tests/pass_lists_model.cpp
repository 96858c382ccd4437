// Host model of the lists of an edge-list call (mdet_amd/csrc/pass_lists.h):
// tiles reserve slots and records, the refinement writes the records of the
// tiles that got a slot and fit, readers go by records_written.  Prints what
// tests/test_pass_lists.py checks.
#include <cstdio>
#include <random>
#include <vector>

#include "../mdet_amd/csrc/pass_lists.h"

using namespace mdet;

int main() {
    std::mt19937_64 rng(7);
    auto below = [&](uint64_t n) { return n ? rng() % n : 0; };
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
    std::printf("reads %ld unwritten_read %ld gaps %ld refused_whole %ld\n", reads, unwritten_read, gaps, refused_whole);
    return 0;
}
