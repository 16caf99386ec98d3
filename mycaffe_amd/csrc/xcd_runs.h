// Tiles of two products in one launch, dealt to the eight XCDs.
#pragma once
#include <algorithm>

namespace mch {

// Workgroup i is on XCD i % 8.  XCD x takes tiles first[x] .. first[x + 1] - 1 of a list that has the tiles of the longer contraction first:
// one run each, so that an XCD's L2 holds the operands of few tiles, and runs of equal work, so that the long tiles are not left to the
// first ones (256 rows, 256 to 1024 values, double: 256 tiles of 1024 k on two XCDs beside 1024 of 256 k on six 18.2 us, so 10.9).
struct XcdRuns { int first[9]; };

// `most`: the longest run, which the launch has eight times
inline XcdRuns xcd_runs(long long tilesLong, int costLong, long long tilesShort, int costShort, int* most)
{
    XcdRuns r;
    const long long longs = tilesLong * costLong, all = longs + tilesShort * costShort;
    *most = 0;
    for (int x = 0; x <= 8; x++) {
        const long long work = all * x / 8;
        r.first[x] = (int)(x == 8 ? tilesLong + tilesShort : work < longs ? (work + costLong - 1) / costLong : tilesLong + (work - longs + costShort - 1) / costShort);
        if (x > 0) *most = std::max(*most, r.first[x] - r.first[x - 1]);
    }
    return r;
}

}  // namespace mch
