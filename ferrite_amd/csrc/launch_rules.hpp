// Arithmetic that host and device have to agree on, or that a test has to see as the library has it: how the passes of the
// streamed tiled kernels are dealt out to blocks.  Plain C++, compiled for the device, the launchers and a host-side test.
#pragma once
#include <stddef.h>

#include "numerics.hpp"

namespace fe {

constexpr int ST_CUS = 256;           // blocks of a launch that goes through several passes per block: one per CU
constexpr int ST_MAX_PASSES = 128;    // entries of a block's table of passes

// Item groups of a unit where blocks go through several passes: raised from a wave per item as far as that leaves the rounds
// of passes the same, so that the last round is not nearly empty (at 509 tokens of the decode shape 136 units x 6 groups
// are 3.2 rounds, x 7 are 3.7).
FE_HD int stream_raise(int n_units, int groups, int items) {
    const int rounds = (n_units * groups + ST_CUS - 1) / ST_CUS;
    int raised = rounds * ST_CUS / n_units;
    if (raised > 2 * groups) raised = 2 * groups;
    if (raised > items) raised = items;
    return raised > groups ? raised : groups;
}

// Blocks of a launch: a multiple of 8, of ST_CUS with several passes each.  Raised groups still fit the rounds that
// max_units * groups passes fill, so every ST_MAX_PASSES of those rounds ask for ST_CUS blocks.
inline unsigned stream_blocks(bool several, int max_units, int groups) {
    const size_t passes = (size_t)max_units * groups;
    if (!several) return (unsigned)((passes + 7) / 8 * 8);
    const size_t table = (size_t)ST_CUS * ST_MAX_PASSES;
    return (unsigned)(ST_CUS * ((passes + table - 1) / table));
}

// The passes of block b of `blocks`: first, first + step, ...  The hardware deals consecutive blocks round-robin over 8 XCDs;
// the passes are cut into 8 contiguous ranges, one per XCD, and block b is number b / 8 of its XCD's.
struct StreamShare {
    int first, step, count;
};
FE_HD StreamShare stream_share(int total, int blocks, int b) {
    const int per_xcd = (total + 7) >> 3, xcd = b & 7, slot = b >> 3, step = blocks >> 3;
    const int left = total - xcd * per_xcd, range = left < per_xcd ? left : per_xcd;
    return StreamShare{xcd * per_xcd + slot, step, slot < range ? (range - slot + step - 1) / step : 0};
}

}  // namespace fe
