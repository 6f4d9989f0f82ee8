// The spread's work lists (pg_worklist.h) on the CPU: the packing of 3-D items
// over the whole range of entries, the bound on the partial slots, the check
// of a 2-D list against lists that are wrong, and the runs of launches.
#include "../../powergrid_amd/csrc/pg_worklist.h"

#include <cstdio>
#include <initializer_list>

struct Item {
    int x, y, z, w;
};

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
    // three patches of 5, 0 and 130 entries, items of up to 64
    const std::vector<long long> cnt = {0, 5, 5, 135};
    const std::vector<Item> good = {{2, 69, 102, -1}, {0, 0, 5, -1}, {-1, 0, 0, -1}, {1, 5, 5, -1},
                                    {2, 5, 69, -1},   {2, 102, 135, -1}};
    auto ok = [&](const std::vector<Item>& v) {
        return spread_items_tile(v.data(), v.size(), cnt, 64);
    };
    CHECK(ok(good));
    auto with = [&](size_t k, Item it) {
        std::vector<Item> v = good;
        v[k] = it;
        return v;
    };
    CHECK(!ok(with(0, {2, 68, 101, -1})));   // an overlap matched by a gap
    CHECK(!ok(with(0, {2, 69, 101, -1})));   // a gap
    CHECK(!ok(with(0, {2, 68, 102, -1})));   // an overlap
    CHECK(!ok(with(1, {0, 0, 6, -1})));      // past the patch
    CHECK(!ok(with(1, {-1, 0, 0, -1})));     // a patch's entries missing
    CHECK(!ok(with(3, {-1, 0, 0, -1})));     // an empty patch without an item
    CHECK(!ok(with(4, {2, 5, 70, -1})));     // longer than an item may be
    CHECK(!ok(with(4, {3, 5, 69, -1})));     // no such patch
    // runs of at most 2^32 - 1 threads that take every block once, in order
    for (int threads : {256, 512})
        for (int times : {1, 7, 96, 1 << 20})
            for (int n : {8, 4096, 1 << 20, (1 << 24) + 8}) {
                long long next = 0;
                bool good = true;
                block_runs(n, times, threads, [&](int o, int k) {
                    good = good && o == next && k > 0 && k % 8 == 0 &&
                           ((long long)k * times * threads < 1LL << 32 || k == 8);
                    next = o + k;
                });
                CHECK(good && next == n);
            }
    for (int threads : {256, 512})
        for (long long blocks : {1LL, 35000LL, 300000LL, 1LL << 22})
            for (int nc : {1, 3, 8, 37, 512, 100000}) {
                long long next = 0;
                bool good = true;
                coil_runs(nc, blocks, threads, [&](int c, int k) {
                    good = good && c == next && k > 0 && k * blocks * threads < 1LL << 32;
                    next = c + k;
                });
                CHECK(good && next == nc);
            }
    std::printf("ok\n");
    return 0;
}
