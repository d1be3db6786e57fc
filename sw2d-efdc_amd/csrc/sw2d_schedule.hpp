// sw2d_schedule.hpp -- the layout of a batch's launch: the order of its blocks
// and the LDS that caps its resident waves.  Host code, standard library only.
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
// ledger waves, which are chains of loads, start first (24 grids of 128^2..1024^2
// in FP64 134.5 us a launch with the clock waves alone there, 134.1 with both; 48
// in FP32 108.4 and 108.2).
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

// LDS to reserve, unused, beside the `own` bytes of a one-wave block so that at
// most `cap` blocks are resident per SIMD (four SIMDs per CU), and no fewer than
// the allocation's steps allow; 0 for no cap.  per_cu, per_block: the LDS of a CU
// and the most that one block may have.  A block's LDS is allocated in steps of
// 1280 bytes (measured: 13568 bytes a block leave 11 on a CU of 160 KiB, not the
// 12 of the quotient; 12800 leave 12).
constexpr size_t kLdsStep = 1280;
inline size_t lds_pad(size_t per_cu, size_t per_block, size_t own, int cap)
{
    if (cap <= 0) return 0;
    // the fewest steps of which 4 cap + 1 blocks no longer fit
    const size_t want = (per_cu / (4 * (size_t)cap + 1) / kLdsStep + 1) * kLdsStep;
    const size_t all = std::min(want, per_block);
    return all > own ? all - own : 0;
}

}  // namespace sw2d
