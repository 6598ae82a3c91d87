// Counts and indexes near 2^32 (pale_common.h) against 64-bit arithmetic: the
// workgroups of a launch, the whole vectors of a scan, the steps of a strided
// loop.
#include <cstdio>

#include "pale_common.h"

int main() {
    const uint32_t top = 0xFFFFFFFFu;
    for (uint32_t n : {0u, 1u, 255u, 256u, 257u, top - 16384u, top - 16383u, top - 256u, top - 4u, top - 1u, top})
        for (uint32_t d : {1u, 3u, 256u, 16384u, 16776960u}) {
            if (pale::ceilDiv(n, d) != ((uint64_t)n + d - 1u) / d) return std::printf("FAIL ceilDiv %u %u\n", n, d), 1;
            for (uint64_t back = 0; back < 40; ++back) {
                const uint32_t i = (uint32_t)(n - back);  // below, at and (wrapped) beyond n
                if (pale::wholeFour(i, n) != ((uint64_t)i + 4u <= n)) return std::printf("FAIL wholeFour %u %u\n", i, n), 1;
            }
            for (uint32_t first : {0u, 7u, n / 2u, n - 1u}) {
                if (n < 64u || d < n / 100000u) continue;
                uint64_t want = first;
                uint32_t i = first;
                while (true) {
                    const bool more = pale::nextItem(i, d, n);
                    want += d;
                    if (more != (want < n)) return std::printf("FAIL nextItem %u %u %u\n", first, d, n), 1;
                    if (!more) break;
                    if (i != want) return std::printf("FAIL nextItem at %u\n", i), 1;
                }
            }
        }
    std::printf("ok\n");
    return 0;
}
