// Tiles of two products in one launch, dealt to the eight XCDs.
#pragma once
#include <algorithm>

namespace mch {

// Workgroup i is on XCD i % 8.  XCD x takes tiles first[x] .. first[x + 1] - 1 of a list that has the tiles of the longer contraction first:
// one run each, so that an XCD's L2 holds the operands of few tiles, and runs of equal work, so that the long tiles are not left to the
// first ones (256 rows, 256 to 1024 values, double: 256 tiles of 1024 k on two XCDs beside 1024 of 256 k on six 17.3 us, so 11.4).
// Where every tile has a CU to itself nothing is to be balanced: they go by count, so that tiles next to each other read the same operands
// (727 rows, 94 to 84, float: 9.2 us, by work 9.8; 1443 rows, 40 to 208 12.3, 12.7).  Where the CUs hold all tiles at once, three to a CU, a run
// longer than an XCD holds has to wait for the first tiles to end.  Tiles of about the same length go by count there too (1.4: 451 rows, 648 to
// 652, 1.37, 13.5 us, by work 15.4; double, 2507 rows, 30 to 3118, 1.23, 36.6, 46.3; but 3387 rows, 52 to 1780, 1.86, 38.3, 26.6), and where the
// short ones are a single stage of 64 k, mostly waiting, no run is longer than that (34 rows, 2986 to 179 6.7 us, by work 8.6; with longer ones
// a second round costs less than long tiles close together: 2655 rows, 226 to 333 46.6, by work 26.6).
struct XcdRuns { int first[9]; };
constexpr int XCD_CUS = 32, XCD_ROOM = 3 * XCD_CUS;   // by the LDS of a workgroup (48 KB)

// `ends`: what a tile costs beside its contraction, in k.  `most`: the longest run, which the launch has eight times
inline XcdRuns xcd_runs(long long tilesLong, int kLong, long long tilesShort, int kShort, int ends, int* most)
{
    XcdRuns r;
    const long long total = tilesLong + tilesShort;
    const bool fits = total <= 8 * XCD_ROOM, byCount = total <= 8 * XCD_CUS || (fits && 5ll * (kLong + ends) < 7ll * (kShort + ends));
    const int costLong = byCount ? 1 : kLong + ends, costShort = byCount ? 1 : kShort + ends;
    const long long longs = tilesLong * costLong, all = longs + tilesShort * costShort;
    for (int x = 0; x <= 8; x++) {
        const long long work = all * x / 8;
        r.first[x] = (int)(x == 8 ? total : work < longs ? (work + costLong - 1) / costLong : tilesLong + (work - longs + costShort - 1) / costShort);
    }
    if (fits && kShort <= 64)
        for (int x = 7; x > 0; x--) r.first[x] = std::max(r.first[x], r.first[x + 1] - XCD_ROOM);
    *most = 0;
    for (int x = 0; x < 8; x++) *most = std::max(*most, r.first[x + 1] - r.first[x]);
    return r;
}

}  // namespace mch
