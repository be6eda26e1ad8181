// Arithmetic that host and device have to agree on, or that a test has to see as the library has it: how the passes of the
// streamed tiled kernels are dealt out to blocks.  Plain C++, compiled for the device, the launchers and a host-side test.
#pragma once
#include <stddef.h>

#include "numerics.hpp"

namespace fe {

constexpr int ST_CUS = 256;           // blocks of a launch that goes through several passes per block: one per CU
constexpr int ST_MAX_PASSES = 128;    // entries of a block's table of passes

// Item groups of the routed experts' units, which come first, and of the shared expert's.  A pass is an item group of a unit;
// the two have groups of their own because the gate/up GEMM of a shared expert of another width has another number of items.
// (With the groups of the wider one for all, most passes of the other had idle waves or nothing to do, at full length.  Layer,
// us, one number / two: 64 experts, top-6, hidden 4096, inter 1024, shared 4096, one term 300 tokens 283 / 206, 4096 tokens
// 1246 / 810; hidden 2048, inter 1408, shared 2816, 2048 tokens one term 343 / 264, two terms 465 / 377.)
struct StreamSplit {
    int routed, shared, groups_r, groups_s;
};
FE_HD int stream_passes(const StreamSplit& s) { return s.routed * s.groups_r + s.shared * s.groups_s; }

// Where blocks go through several passes the groups, a wave per item at first, are raised as far as that leaves the rounds of
// passes the same, so that the last round is not nearly empty (at 509 tokens of the decode shape 136 units x 6 groups are
// 3.2 rounds, x 7 are 3.7).
FE_HD StreamSplit stream_raise(StreamSplit s, int items_r, int items_s) {
    const int passes = stream_passes(s), rounds = (passes + ST_CUS - 1) / ST_CUS;
    const int more = (rounds * ST_CUS - passes) / (s.routed + s.shared);
    auto raise = [&](int groups, int items) {
        int g = groups + more;
        if (g > 2 * groups) g = 2 * groups;
        if (g > items) g = items;
        return g > groups ? g : groups;
    };
    s.groups_r = raise(s.groups_r, items_r);
    s.groups_s = raise(s.groups_s, items_s);
    return s;
}

// Blocks of a launch sized for `most` units: a multiple of 8, of ST_CUS with several passes each.  Raised groups still fit the
// rounds that the passes of those units fill, so every ST_MAX_PASSES of the rounds ask for ST_CUS blocks.
inline unsigned stream_blocks(bool several, const StreamSplit& most) {
    const size_t passes = (size_t)most.routed * most.groups_r + (size_t)most.shared * most.groups_s;
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
