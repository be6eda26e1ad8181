// Arithmetic that host and device have to agree on, or that a test has to see as the library has it: how the passes of the
// streamed tiled kernels are dealt out to blocks, and which form of the f32 expert kernels a call takes.  Plain C++, compiled
// for the device, the launchers and the tests.
#pragma once
#include <stddef.h>

#include "numerics.hpp"

namespace fe {

// Units of up to unit_rows rows that a call may have: what tables and grids are sized for.
inline int max_units_for(int n, int topk, int n_experts, int has_shared, int unit_rows) {
    long assign = (long)n * topk;
    long active_max = assign < n_experts ? assign : n_experts;
    long u = assign / unit_rows + active_max + (has_shared ? (n + unit_rows - 1) / unit_rows : 0);
    return (int)u;
}

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
    int first, step, left;   // left: passes of the XCD's range from first on, <= 0 for none
};
FE_HD StreamShare stream_share(int total, int blocks, int b) {
    const int per_xcd = (total + 7) >> 3, xcd = b & 7, slot = b >> 3;
    const int left = total - xcd * per_xcd;
    return StreamShare{xcd * per_xcd + slot, blocks >> 3, (left < per_xcd ? left : per_xcd) - slot};
}
FE_HD int stream_count(const StreamShare& s) { return s.left > 0 ? (s.left + s.step - 1) / s.step : 0; }

// The f32 expert kernels: one pair of tiles per wave (0), or per block of four waves where the former leaves some of the chip's
// 1024 SIMDs without work (1) and where its last round of waves is so empty that rounds x blocks of 128 k per wave come out a
// tenth larger (2: a few thousand waves; beyond that the rounds even out and the split only stages the activations four times
// as often).  max_units is what the grid is sized for, the live units are estimated; rows, sh_rows and K: weight rows of a
// routed and of the shared expert and the reduction length.  Kernel, us, a wave / a block per pair: gate/up of hidden 2880,
// inter 480, 64 experts, 9 tokens 101 / 65, 64 tokens 106 / 92; hidden 2880, 32 experts 75.3 / 63.9; on the other side hidden
// 2080, inter 736, 27 tokens 57.6 / 59.6, its down 31.4 / 31.7; 64 experts, inter 1056 104.7 / 112.3; layer of hidden 1440,
// 64 experts, 64 tokens 87.8 / 92.9.
inline int f32_split(int n, int topk, int n_experts, int max_units, int rows, int sh_rows, int K, bool down) {
    const int step = down ? 32 : 16;   // output rows per pair of tiles
    if ((long)max_units * ((rows > sh_rows ? rows : sh_rows) / step) <= 1024) return 1;
    const double E = n_experts, hit = E * (1.0 - pow(1.0 - topk / E, n)), per_expert = n * (double)topk / hit;
    const double waves = hit * fmax(1.0, per_expert / 16.0 + 0.5) * (rows / step) + (sh_rows > 0 ? (n + 15) / 16 : 0) * (double)(sh_rows / step);
    const int kblocks = (K + 127) / 128;
    // whole rounds without the split, on the low side of the estimate; four times as many shorter ones fill up half of their last
    const double whole = ceil(0.97 * waves / 1024.0) * kblocks, split = (4.0 * waves / 1024.0 + 0.5) * ((kblocks + 3) / 4);
    return waves <= 4096.0 && split <= 0.9 * whole ? 2 : 0;
}

}  // namespace fe
