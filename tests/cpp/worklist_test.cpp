// The spread's work lists (pg_worklist.h) on the CPU: the packing of 3-D items
// over the whole range of entries and the bound on the partial slots.
#include "../../powergrid_amd/csrc/pg_worklist.h"

#include <cstdio>
#include <initializer_list>

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);       \
            return 1;                                         \
        }                                                     \
    } while (0)

int main()
{
    using namespace pg;
    // first entries around every power of two up to the limit
    for (int b = 0; b <= 38; ++b)
        for (long long d = -1; d <= 1; ++d) {
            const long long first = (1LL << b) + d;
            if (first < 0 || first >= kP3MaxEntries) continue;
            for (long long n : {0LL, 1LL, 255LL, (long long)p3_part_entries(kP3MaxEntries)}) {
                const int y = p3_y(first), z = p3_z(first, n);
                CHECK(p3_count(z) == n && p3_first(y, z) == first);
            }
        }
    // parts of at least 256 entries, at most 65536 of them however they lie
    CHECK(p3_part_entries(0) == 256 && p3_part_entries(256LL * 32768) == 256);
    for (long long total = 1000; total < kP3MaxEntries; total *= 7) {
        const long long t = p3_part_entries(total);
        // all in one patch, or in patches one entry too heavy
        CHECK((total + t - 1) / t <= 65536 && 2 * (total / (t + 1)) <= 65536);
    }
    std::printf("ok\n");
    return 0;
}
