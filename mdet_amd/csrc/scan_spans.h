// Column spans of the first pass's items: by size, and the ones the autotuner
// tries (host code of tnf_pairs.hip).
#pragma once

#include <cstdint>
#include <vector>

namespace mdet {

// Default column span by size: the power of two nearest n / 50 in [512, 16384].
// Longer spans spare the box scan row fragments and boxes (43 -> 34 us at 50,000
// contigs and 10.64 -> 10.49 ms at 1,000,000 against n / 100 and at most 4096);
// short ones keep enough items for the blocks of small inputs.
inline uint32_t seg_cols_for(uint32_t n) {
    uint32_t seg = 512;
    while (seg < 16384 && (uint64_t)seg * 3 / 2 * 50 < n) seg *= 2;
    return seg;
}

// Spans to time at n contigs: the default, then the other powers of two from
// 512 to 4096, or on to the default where it is longer.
inline std::vector<uint32_t> tune_spans(uint32_t n) {
    const uint32_t by_size = seg_cols_for(n);
    std::vector<uint32_t> spans{by_size};
    for (uint32_t seg = 512; seg <= 4096 || seg <= by_size; seg *= 2)
        if (seg != by_size) spans.push_back(seg);
    return spans;
}

// Whether a shape's time replaces the best so far: by more than medians of the
// same shape differ by (1-2%), so that noise does not take the default away.
inline bool tuned_shape_wins(double ms, double best) { return ms < 0.98 * best; }

}  // namespace mdet
