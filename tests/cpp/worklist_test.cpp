// The spread's work lists (pg_worklist.h) on the CPU: the bound on the partial
// slots.
#include "../../powergrid_amd/csrc/pg_worklist.h"

#include <cstdio>

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
    // parts of at least 256 entries, at most 65536 of them however they lie
    CHECK(p3_part_entries(0) == 256 && p3_part_entries(256LL * 32768) == 256);
    for (long long total = 1000; total < 1LL << 38; total *= 7) {
        const long long t = p3_part_entries(total);
        // all in one patch, or in patches one entry too heavy
        CHECK((total + t - 1) / t <= 65536 && 2 * (total / (t + 1)) <= 65536);
    }
    std::printf("ok\n");
    return 0;
}
