// The order in which attention over prompts takes its workgroups, a tile of 128 (token, head) rows of a sequence and kv head each.
#pragma once
#include "common.h"

// The kv heads lie side by side, so that a kv head's workgroups are on one XCD (on 8 / heads of them, `side` tiles in a row, where the
// heads are 4, 2 or 1), whose L2 then holds its keys and values, and tiles go from the last (most keys) on: over all sequences at once (up to 16
// of them; each row of equal tiles turned by a number of its own, since workgroup numbers fall on shader engines by their low bits, and sequences that
// have no such tile would leave the same ones idle), else sequence by sequence, which then find their keys in the L2 as the tiles
// follow one another.  Where all workgroups are resident at once, two to a compute unit, those of the second round (from `fold` on) are taken from
// the last on: a long and a short one share a unit.  Other numbers of heads: a kv head's tiles in a row, every second half of the heads from
// the first tile on where all are resident (`fold` 1).  us before (a kv head's tiles in a row) and now, 32 heads of 128 over 8: 2,048
// tokens 65.5 / 61.6, 4,096 234 / 167, 7,001 (window 4,096) 450 / 384, 16,384 2,400 / 2,330, four times 2,000 215 / 170, eight times 1,000
// 155 / 106, 16 times 500 114 / 74, 1,357 to 93 75 / 69, 3,000 and 1,000 137 / 106 (unturned 162), 1,000 and five times 50 34.1 / 35.0, 64 times 150
// 60.5 / 59.3 (over all at once 66), 32 times 200 46.9 / 44.9 (50.6); 32 over 4 heads of 64, 3,000 and 1,000 90 / 71; 32 over 2, 2,000, 1,500 and
// 700 89 / 79.
struct PrefillOrder {
    int heads, B, tiles, side, fold, by_tile;
    __device__ __forceinline__ void place(int& head, int& b, int& tile) const {
        int id = blockIdx.y * gridDim.x + blockIdx.x;
        if (!side) {
            tile = tiles - 1 - id % tiles;
            id /= tiles;
            head = id % heads;
            b = id / heads;
            if (fold && ((head * 2 / heads) & 1)) tile = tiles - 1 - tile;
            return;
        }
        head = id % heads;
        int u = id / heads;
        if (u >= fold) u = fold + tiles * B - 1 - u;
        const int lo = u % side, rows = tiles / side;
        u /= side;
        const int hi = by_tile ? u / B : u % rows;
        b = by_tile ? (u + hi + __popc(hi)) % B : u / rows;
        tile = tiles - 1 - (hi * side + lo);
    }
};

// For sequences of up to `rows` rows and workgroups of 256 threads, of which `each` fit a compute unit; the grid's x, 0 where the grid is too large.
// Its y is B: workgroups are numbered along x first, and a launch's 2^32 threads hold for x alone.
static inline unsigned prefill_order(PrefillOrder& o, long long rows, int heads, int B, int cus, int each) {
    const int side = heads % 8 == 0 ? 1 : 8 % heads == 0 ? 8 / heads : 0;
    long long tiles = (rows + 127) / 128;
    if (side) tiles = (tiles + side - 1) / side * side;
    if (tiles > 0xffffff || tiles * heads > 0xffffff || tiles * heads * B > 0x7fffffffLL) return 0;
    const bool resident = each == 2 && cus > 0 && tiles * B * heads <= 2LL * cus;
    o = {heads, B, (int)tiles, side, side ? (resident && cus % heads == 0 ? cus / heads : (int)(tiles * B)) : resident, B <= 16};
    return (unsigned)(tiles * heads);
}
