// Tiles of two products in one launch, dealt to the eight XCDs.
#pragma once
#include <algorithm>

namespace mch {

// Workgroup i is on XCD i % 8.  XCD x takes tiles first[x] .. first[x + 1] - 1 of a list that has the tiles of the longer contraction first:
// one run each, so that an XCD's L2 holds the operands of few tiles, and runs of equal work, so that the long tiles are not left to the
// first ones (256 rows, 256 to 1024 values, double: 256 tiles of 1024 k on two XCDs beside 1024 of 256 k on six 17.3 us, so 11.4).
// Where every tile has a CU to itself nothing is to be balanced: they go by count, so that tiles next to each other read the same operands
// (727 rows, 94 to 84, float: 9.2 us, by work 9.8; 1443 rows, 40 to 208 12.5, 12.8).  Where the CUs hold all tiles at once, three to a CU, they
// do too if the long ones are less than twice the short ones (double, 993 rows, 48 to 1546 13.6 us, 14.3; 40 rows, 384 to 1536, thirteen times
// as long, float, 12.5 us, by work 12.0), and no XCD is given more than it holds: the rest would wait for the first to end (34 rows, 2986 to
// 179: 94 tiles each 6.7 us, 123 short ones on some 8.6; 451 rows, 648 to 652 13.5, 15.4; double, 2507 rows, 30 to 3118 36.9, 46.3).
struct XcdRuns { int first[9]; };
constexpr int XCD_CUS = 32, XCD_ROOM = 3 * XCD_CUS;   // by the LDS of a workgroup (48 KB)

// `most`: the longest run, which the launch has eight times
inline XcdRuns xcd_runs(long long tilesLong, int costLong, long long tilesShort, int costShort, int* most)
{
    XcdRuns r;
    const long long total = tilesLong + tilesShort;
    if (total <= 8 * XCD_CUS || (total <= 8 * XCD_ROOM && costLong < 2 * costShort)) costLong = costShort = 1;
    const long long longs = tilesLong * costLong, all = longs + tilesShort * costShort;
    for (int x = 0; x <= 8; x++) {
        const long long work = all * x / 8;
        r.first[x] = (int)(x == 8 ? total : work < longs ? (work + costLong - 1) / costLong : tilesLong + (work - longs + costShort - 1) / costShort);
    }
    if (total <= 8 * XCD_ROOM)
        for (int x = 7; x > 0; x--) r.first[x] = std::max(r.first[x], r.first[x + 1] - XCD_ROOM);
    *most = 0;
    for (int x = 0; x < 8; x++) *most = std::max(*most, r.first[x + 1] - r.first[x]);
    return r;
}

}  // namespace mch
