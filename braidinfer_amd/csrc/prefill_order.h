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
// 155 / 106, 16 times 500 114 / 74, 1,357 to 93 75 / 69, 3,000 and 1,000 137 / 106 (unturned 162), 1,000 and five times 50 34.1 / 34.9, 64 times 150
// 60.5 / 59.3 (over all at once 66), 32 times 200 46.9 / 44.9 (50.6); 32 over 4 heads of 64, 3,000 and 1,000 90 / 71; 32 over 2, 2,000, 1,500 and
// 700 89 / 79.
//
// Nothing is divided that the grid can hold: five divisions a workgroup cost short prompts 0.4 us (67 tokens 8.9 and 8.6 without, 512 20.1 and 19.6, as before the order).
struct PrefillOrder {
    int B, tiles, total, side, shift, fold, by_tile;         // total: tiles of all sequences; side = 1 << shift, or 0
    __device__ __forceinline__ void place(int& head, int& b, int& tile) const {
        if (!side) {                                         // grid (tiles, heads, B)
            head = blockIdx.y;
            b = blockIdx.z;
            tile = fold && ((head * 2 / (int)gridDim.y) & 1) ? (int)blockIdx.x : tiles - 1 - (int)blockIdx.x;
            return;
        }
        head = blockIdx.x;                                   // grid (heads, a run of all tiles, runs)
        int u = blockIdx.z * gridDim.y + blockIdx.y;
        b = 0;
        tile = tiles;                                        // none
        if (u >= total) return;
        if (u >= fold) u = fold + total - 1 - u;
        if (B > 1) {
            const int lo = u & (side - 1);
            u >>= shift;
            const int hi = by_tile ? u / B : u % (tiles >> shift);
            b = by_tile ? (u + hi + __popc(hi)) % B : u / (tiles >> shift);
            u = (hi << shift) + lo;
        }
        tile = tiles - 1 - u;
    }
};

// For sequences of up to `rows` rows and workgroups of which `each` fit a compute unit; false where there are too many.
static inline bool prefill_order(PrefillOrder& o, dim3& grid, long long rows, int heads, int B, int cus, int each) {
    const int shift = heads % 8 == 0 ? 0 : heads == 4 ? 1 : heads == 2 ? 2 : heads == 1 ? 3 : -1;
    long long tiles = (rows + 127) / 128;
    if (shift > 0) tiles = (tiles + (1 << shift) - 1) >> shift << shift;
    if (tiles > 0xffffff || tiles * B > 0x7fffffffLL) return false;
    const bool resident = each == 2 && cus > 0 && tiles * B * heads <= 2LL * cus;
    const int total = (int)(tiles * B), run = total < 32768 ? total : 32768;
    o = {B, (int)tiles, total, shift < 0 ? 0 : 1 << shift, shift, shift < 0 ? resident : resident && cus % heads == 0 ? cus / heads : total, B <= 16};
    grid = shift < 0 ? dim3((unsigned)tiles, heads, B) : dim3(heads, run, (total - 1) / run + 1);
    return true;
}
