// Prints seg_cols_for and tune_spans (mdet_amd/csrc/scan_spans.h) for
// tests/test_scan_spans.py: n, default, spans.
#include <cstdio>

#include "../mdet_amd/csrc/scan_spans.h"

int main() {
    for (uint64_t n = 6145; n < 1u << 30; n = n * 5 / 4) {
        std::printf("%llu %u", (unsigned long long)n, mdet::seg_cols_for((uint32_t)n));
        for (uint32_t s : mdet::tune_spans((uint32_t)n)) std::printf(" %u", s);
        std::printf("\n");
    }
    std::printf("%d %d\n", mdet::tuned_shape_wins(0.99, 1.0), mdet::tuned_shape_wins(0.9, 1.0));
    return 0;
}
