// pg_worklist.h -- the spread's work lists: how many entries an
// item of the 3-D list takes.  Plain C++.
#pragma once

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

}  // namespace pg
