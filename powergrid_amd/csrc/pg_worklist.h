// pg_worklist.h -- the gridding's work lists: how an item of the 3-D spread's
// list is packed, whether a 2-D list takes every entry once, and how lists go
// in launches.  Plain C++ besides the device attributes.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

#ifdef __HIPCC__
#define PG_HD __host__ __device__
#else
#define PG_HD
#endif

namespace pg {

// 3-D spread: entries of a patch summed by one wavefront.  A lone wavefront
// takes about 500 clocks per 4 entries, so 256 of them (14 us) keep the
// longest item short against the whole launch.  A plan of many entries takes
// longer items, 1/32768 of them all: still many to a wavefront of the chip, and
// at most 65536 partial slots (1 GB for 32 grids; a slot for every 256 entries
// would be more than the samples' values).
constexpr int kP3Entries = 256;
inline int p3_part_entries(long long total)
{
    const long long n = (total + 32767) / 32768;
    return n > kP3Entries ? (int)n : kP3Entries;
}

// Its items are {patch or -1, y, z, slot or -1} with the first entry and the
// number of entries in y and z.  A sample has up to 64 entries, so a plan can
// hold more than 32 bits count: y and the upper 8 bits of z are the first
// entry, the lower 24 bits of z the number (p3_part_entries() at most).
constexpr long long kP3MaxEntries = 1LL << 38;
inline int p3_y(long long first) { return (int)(uint32_t)first; }
inline int p3_z(long long first, long long n) { return (int)(uint32_t)(n | first >> 32 << 24); }
PG_HD inline int p3_count(int z) { return z & 0xFFFFFF; }
PG_HD inline long long p3_first(int y, int z)
{
    return (long long)(uint32_t)y | (long long)((uint32_t)z >> 24) << 32;
}

// Whether the 2-D items {patch or -1, first entry, end, slot} hold every
// entry of patch q, cnt[q] .. cnt[q + 1], once, at most `longest` to an item,
// and name every patch.  The patches' entries follow each other, so the items
// lie within their patches and together tile 0 .. cnt[np].
template <class Item>
bool spread_items_tile(const Item* items, size_t n, const std::vector<long long>& cnt, int longest)
{
    const long long np = (long long)cnt.size() - 1;
    std::vector<int> step((size_t)cnt[np] + 1, 0);  // changes of the cover count
    std::vector<char> met((size_t)np, 0);
    for (size_t k = 0; k < n; ++k) {
        const Item& it = items[k];
        if (it.x < 0) continue;
        if (it.x >= np || it.z < it.y || it.z - it.y > longest || it.y < cnt[it.x] ||
            it.z > cnt[it.x + 1])
            return false;
        ++step[it.y];
        --step[it.z];
        met[it.x] = 1;
    }
    int cover = 0;
    for (long long e = 0; e < cnt[np]; ++e)
        if ((cover += step[e]) != 1) return false;
    for (char m : met)
        if (!m) return false;
    return true;
}

// blocks of `threads` threads that one launch can have (its threads in 32
// bits: with more, a part of them runs and no error is given)
constexpr int max_blocks(int threads) { return (int)(((1LL << 32) - 1) / threads); }

// launch(first, count) over a work list of n blocks (a multiple of 8), each
// `times` times, in runs that one launch can have; every run a multiple of 8
// blocks, one for each XCD
template <class F>
void block_runs(int n, int times, int threads, F launch)
{
    const int fit = max_blocks(threads) / times / 8 * 8;
    const int run = fit > 8 ? fit : 8;
    for (int o = 0; o < n; o += run) launch(o, n - o < run ? n - o : run);
}

// the same over nc coils of `blocks` blocks each; a multiple of 8 coils at a
// time, which keep their XCDs, where that many fit
template <class F>
void coil_runs(int nc, long long blocks, int threads, F launch)
{
    const long long fit = max_blocks(threads) / blocks;
    const int run = fit >= nc ? nc : fit >= 8 ? (int)(fit / 8 * 8) : fit > 1 ? (int)fit : 1;
    for (int c = 0; c < nc; c += run) launch(c, nc - c < run ? nc - c : run);
}

}  // namespace pg
