// sw2d_schedule.hpp -- the order of the blocks of a batch's launch.  Host code,
// standard library only.
#pragma once
#include <stddef.h>

#include <algorithm>
#include <vector>

namespace sw2d {

// one block of a batched launch: scenario and block within it
struct TileRef {
    int sid, local;
};

// bookkeeping waves besides those of the lake-inflow records (64 each): the
// clock and the forcing, the ledger
constexpr int kBookParts = 2;
inline int book_blocks(int nbc) { return kBookParts + (nbc + 63) / 64; }

// the launch's tile table: each member's blocks in a run (order 0), or the
// members interleaved block by block (order 1), so that every stretch of
// the launch holds tiles of many members.  Either way the members' clock and
// ledger waves, which are chains of loads, start first.
inline void order_tiles(const std::vector<int> &counts, const std::vector<int> &sids, int order,
                        std::vector<TileRef> &tiles)
{
    tiles.clear();
    if (order == 0) {
        for (int i = 0; i < kBookParts; i++)
            for (size_t m = 0; m < counts.size(); m++) tiles.push_back(TileRef{sids[m], i});
        for (size_t m = 0; m < counts.size(); m++)
            for (int i = kBookParts; i < counts[m]; i++) tiles.push_back(TileRef{sids[m], i});
        return;
    }
    int most = 0;
    for (int c : counts) most = std::max(most, c);
    for (int i = 0; i < most; i++)
        for (size_t m = 0; m < counts.size(); m++)
            if (i < counts[m]) tiles.push_back(TileRef{sids[m], i});
}

}  // namespace sw2d
