// Plain-data kernel arguments, filled by the C-ABI entry points after validation.
#pragma once

#include <stdint.h>

#include "chill_mask.h"

namespace chill {

struct Strides3 {  // element strides of a [B, H, T, D] tensor with unit inner stride
    int64_t b, h, t;
};

// The order in which a launch's workgroups take their (head, tile) items (work_order, chill_tiles.h).
struct WorkOrder {
    int32_t small;    // blocks that come first, of `sets` sets of heads each; the others have 8 more.  0: contiguous runs
    int32_t sets;     // a multiple of 8
    int32_t rest;     // sets of an incomplete round, which go with the first block; + 8: such a block takes its heads in turn
};

struct FwdParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    float* lse;  // nullable
    const int32_t* lens;  // nullable
    Strides3 sq, sk, sv, so;
    int64_t lse_b, lse_h;  // fp32 [B, H, T], unit inner stride
    int64_t lens_stride;
    int32_t B, H, H_kv, T;
    int32_t group;         // H / H_kv
    int32_t order_small;   // the WorkOrder; what only a launch in blocks reads is the struct's end, see order_of
    float scale_log2;      // sm_scale * log2(e)
    MaskArgs margs;
    int32_t order_sets, order_rest;
};

// The forward of a launch with fewer q-tiles than the chip has room for: the keys of the long q-tiles are split into
// parts, each an item of its own (plan_fwd_split, chill_fwd_split.h).  The items of a head, longest first:
// q-tile | part << 10 | parts << 15 | first partial result of the q-tile << 20.
constexpr int kFwdSplitMaxItems = CHILL_FWD_SPLIT_MAX_ITEMS, kFwdSplitMaxQTiles = 256, kFwdSplitMaxParts = 16;
struct FwdSplit {
    float* partials;      // [head][partials_per_head] results of one part each
    int32_t n_items, n_q_tiles, partials_per_head, partial_floats;
    int32_t part_tiles;   // tiles of keys in every part of a q-tile but the last
    uint32_t item[kFwdSplitMaxItems];
    uint32_t merge[kFwdSplitMaxQTiles];  // any item of every q-tile
    uint32_t* again;  // [head][q-tile]: a q-tile of one part whose sums left the range (written for every such q-tile)
};

struct DeltaParams {
    const void* o;
    const void* d_o;
    float* delta;
    Strides3 so, sdo;
    int64_t delta_b, delta_h;
    int32_t B, H, T;
};

struct BwdParams {
    const void* q;
    const void* k;
    const void* v;
    const void* d_o;
    void* dq;
    void* dk;
    void* dv;
    const float* lse;
    const float* delta;
    const int32_t* lens;  // nullable
    // dQ that computes delta itself (chill_bwd_dq_delta): the forward's output, and where the rows of
    // delta = rowsum(O * dO) go for the dK/dV launch that follows; both null otherwise
    const void* o;
    float* delta_out;
    Strides3 sq, sk, sv, sdo, sdq, sdk, sdv, so;
    int64_t lse_b, lse_h;
    int64_t delta_b, delta_h;
    int64_t lens_stride;
    int32_t B, H, H_kv, T;
    int32_t group;
    int32_t order_small;
    float sm_scale;
    float scale_log2;
    MaskArgs margs;
    int32_t order_sets, order_rest;
};

// Three fields side by side cost the banded forward 300 moves of its pointers to vector lanes and back (scalar loads of eight
// words in the middle of the struct leave no room for those of sixteen), and moved the code of the kernels that do not read
// them: SlidingWindow(16, 16) from cold caches, fp16 B8 H4 T6000 D128 61 -> 64 us, fp32 B8 H8 T6000 D64 234 -> 242.
template <typename P>
CHILL_HD WorkOrder order_of(const P& p) {
    return WorkOrder{p.order_small, p.order_sets, p.order_rest};
}
template <typename P>
inline void set_order(P& p, WorkOrder order) {
    p.order_small = order.small;
    p.order_sets = order.sets;
    p.order_rest = order.rest;
}

// One row of the static tile table (the replacement for the reference's autotune tables,
// autotune.py:11-119): rows per workgroup = 32 * waves, streamed tile size.
struct TileConfig {
    int rows;      // resident rows per workgroup (q rows for fwd / dQ, k rows for dK/dV)
    int streamed;  // rows of one streamed tile
    int waves;
    int lds_bytes;
};

}  // namespace chill
