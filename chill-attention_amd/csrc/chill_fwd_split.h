// Split of the long q-tiles of an underfilled forward along their keys: the plan.  The kernels are fwd_split_kernel
// and fwd_merge_kernel (chill_fwd_kernel.h).
#pragma once

#include "chill_params.h"
#include "chill_tiles.h"

namespace chill {

// Shapes: the 16-bit forwards with the generated loop, masks that are not banded (a band's q-tiles are all short).
constexpr bool fwd_split_serves(int mask_id, int D, int dtype) {
    return CHILL_FWD_FAST && dtype != CHILL_F32 && (D == 64 || D == 128) &&
           (mask_id == CHILL_MASK_FULL || mask_id == CHILL_MASK_CAUSAL || mask_id == CHILL_MASK_PREFIX_LM);
}

// What an item costs beyond its 64-key tiles, in the time of one (1.2 us at D = 128 with one workgroup on the CU, 0.56 us
// at D = 64): Q, the first tiles and the result, all workgroups of the launch at once; a part also writes its partial
// result; the second launch, which adds the parts up, is paid once.
constexpr int kFwdItemOverhead = 8, kFwdPartOverhead = 16, kFwdMergeOverhead = 10;

// The plan of a launch of `heads` heads: how many bytes of workspace it takes, 0 if the launch is not split.  A q-tile of
// n tiles of keys is cut into parts of c tiles, the last one what is left (up to half a part's overhead more than c).
// Unequal on purpose: under a causal mask the remainders are as short as the q-tiles at the other end, and longest first
// they fill the CUs the long parts leave (B1 H8 T8192 D128, 32 q-tiles of 4 .. 128 tiles and 32 CUs per head: parts of
// 66 tiles and pairs that add up to 66).  c is the one of longest / 1, 2, .. and of the work per slot whose launch should
// end first.  A launch ends no earlier than its longest item, and than its work over the slots the chip has, where a tile
// takes a third longer (the whole chip at work runs at the board's power limit; 1.6 against 1.2 us); items of one length
// (full mask) run in whole rounds.  Two workgroups share a CU at D = 64, each at about three quarters of its speed alone.
// Split where that saves a twelfth.  Measured, us, bf16, B1, whole -> split:
//   causal  D128  H2 T16384 258 -> 155   H3 T8192 135 -> 84   H4 T8192 135 -> 98   H8 T8192 157 -> 142   H8 T4096 79 -> 69
//           D64   H2 T16384 133 -> 90    H3 T8192  73 -> 44   H4 T8192  66 -> 52   H6 T8192  77 -> 68    H8 T4096 37 -> 33
//   full    D128  H2 T16384 269 -> 232   H3 T8192 135 -> 107  H4 T8192 140 -> 129  H6 T4096  74 -> 66
//   left whole by the rule (measured split): causal D128 H16 T4096 85 (89), H12 T4042 80 (85); full H12 T8192 354 (366), D64
//   H6 T4096 36 (40).
inline int64_t plan_fwd_split(int mask_id, const MaskArgs& margs, int64_t heads, int T, int D, int dtype, void* workspace,
                              FwdSplit* out) {
    if (!fwd_split_serves(mask_id, D, dtype)) return 0;
    const TileConfig cfg = fwd_tile_config(mask_id, D, dtype);
    const int n_q_tiles = cdiv(T, cfg.rows);
    // launches that fill the chip with pairs of q-tiles, and those that other kernels take
    if (n_q_tiles > kFwdSplitMaxQTiles || heads * ((n_q_tiles + 1) / 2) >= kComputeUnits) return 0;
    if (fwd_takes_small(mask_id, heads, T, D, dtype)) return 0;
    if (D == 128 && fwd_takes_short_row(mask_id, kWholeSequence, heads, T)) return 0;
    const int slots = D == 64 ? kComputeUnits * 3 / 2 : kComputeUnits;
    int tiles[kFwdSplitMaxQTiles];
    int longest = 0;
    int64_t all = 0;
    CHILL_DISPATCH_MASK(mask_id, {
        for (int i = 0; i < n_q_tiles; i++) {
            const TileRange r = tile_range<MASK_ID, true>(i * cfg.rows, cfg.rows, cfg.streamed, T, false, margs);
            tiles[i] = r.end > r.start ? r.end - r.start : 0;
            if (tiles[i] > longest) longest = tiles[i];
            all += tiles[i];
        }
    });
    constexpr int kSlack = kFwdPartOverhead / 2;
    auto parts_of = [&](int i, int c) { return tiles[i] > c + kSlack ? cdiv(tiles[i] - kSlack, c) : 1; };
    auto launch_time = [&](int c) -> int64_t {
        int64_t items = 0, work = all;
        bool any = false;
        for (int i = 0; i < n_q_tiles; i++) {
            const int parts = parts_of(i, c);
            any = any || parts > 1;
            items += parts;
            work += parts > 1 ? parts * kFwdPartOverhead : kFwdItemOverhead;
            if (parts > kFwdSplitMaxParts) return INT64_MAX;
        }
        if (items > kFwdSplitMaxItems) return INT64_MAX;
        const int64_t one = any ? c + kFwdPartOverhead : longest + kFwdItemOverhead;
        const int64_t spread = heads * work / slots * 4 / 3;
        const int64_t rounds = mask_id == CHILL_MASK_FULL ? (heads * items + slots - 1) / slots * one : one;
        return (spread > rounds ? spread : rounds) + (any ? kFwdMergeOverhead : 0);
    };
    const int64_t whole = launch_time(longest);
    int best = longest;
    int64_t best_time = whole * 11 / 12;
    auto consider = [&](int c) {
        if (c < kFwdPartOverhead || c >= longest) return;
        const int64_t time = launch_time(c);
        if (time < best_time) {
            best_time = time;
            best = c;
        }
    };
    for (int k = 2; k <= kFwdSplitMaxParts; k++) consider(cdiv(longest, k));
    if (mask_id != CHILL_MASK_FULL) consider((int)(heads * all / slots) + kFwdItemOverhead);
    if (best == longest) return 0;
    // items sorted by their length, longest first
    constexpr int kMostKeyTiles = kFwdSplitMaxQTiles * 256 / 64;  // (q-tiles of at most 256 rows)
    int place[kMostKeyTiles + 1] = {};
    auto last_of = [&](int i) { return tiles[i] - (parts_of(i, best) - 1) * best; };
    for (int i = 0; i < n_q_tiles; i++) {
        place[best] += parts_of(i, best) - 1;
        place[last_of(i)]++;
    }
    int n_items = 0, partials = 0;
    for (int n = longest; n >= 0; n--) {
        const int count = place[n];
        place[n] = n_items;
        n_items += count;
    }
    for (int i = n_q_tiles - 1; i >= 0; i--) {
        const int parts = parts_of(i, best);
        const uint32_t common = i | parts << 15 | partials << 20;
        for (int j = 0; j + 1 < parts; j++) out->item[place[best]++] = common | j << 10;
        out->item[place[last_of(i)]++] = common | (parts - 1) << 10;
        out->merge[i] = common;
        if (parts > 1) partials += parts;
    }
    out->n_items = n_items;
    out->n_q_tiles = n_q_tiles;
    out->partials_per_head = partials;
    out->partial_floats = cfg.rows * D + 2 * cfg.waves * 64;  // O^T; m0 and l of every lane
    out->part_tiles = best;
    const int64_t partial_bytes = heads * partials * out->partial_floats * 4;
    out->partials = static_cast<float*>(workspace);
    out->again = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + partial_bytes);
    return partial_bytes + heads * n_q_tiles * 4;
}

}  // namespace chill
