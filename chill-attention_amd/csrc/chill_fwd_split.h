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

// What an item costs beyond its 64-key tiles, in the time of one: Q, the first tiles and the result; a part also the
// partial result and its share of the sum.
constexpr int kFwdItemOverhead = 4, kFwdPartOverhead = 10;

// The plan of a launch of `heads` heads: how many bytes of workspace it takes, 0 if the launch is not split.  A q-tile of
// n tiles of keys is cut into equal parts of at most c tiles; of the c = longest / 1, 2, .. the one is taken whose
// launch should end first, and only if it saves an eighth.  A launch ends no earlier than its work over the workgroups the
// chip holds at once, and than its longest item; items of one length (full mask) run in whole rounds.
inline int64_t plan_fwd_split(int mask_id, const MaskArgs& margs, int64_t heads, int T, int D, int dtype, void* workspace, FwdSplit* out) {
    if (!fwd_split_serves(mask_id, D, dtype)) return 0;
    const TileConfig cfg = fwd_tile_config(mask_id, D, dtype);
    const int n_q_tiles = cdiv(T, cfg.rows);
    // launches that fill the chip with pairs of q-tiles, and those that other kernels take
    if (n_q_tiles > kFwdSplitMaxQTiles || heads * ((n_q_tiles + 1) / 2) >= kComputeUnits) return 0;
    if (fwd_takes_small(mask_id, heads, T, D, dtype) || (D == 128 && fwd_takes_short_row(mask_id, kWholeSequence, heads, T))) return 0;
    const int slots = kComputeUnits * (D == 64 ? 2 : 1);
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
    int best = 1;
    int64_t best_time = 0;
    for (int k = 1; k <= kFwdSplitMaxParts; k++) {
        const int most = cdiv(longest, k);
        if (most < kFwdPartOverhead && k > 1) break;
        int64_t items = 0, work = all;
        for (int i = 0; i < n_q_tiles; i++) {
            const int parts = tiles[i] > most ? cdiv(tiles[i], most) : 1;
            items += parts;
            work += parts > 1 ? parts * kFwdPartOverhead : kFwdItemOverhead;
        }
        if (items > kFwdSplitMaxItems) break;
        const int64_t one = most + (k > 1 ? kFwdPartOverhead : kFwdItemOverhead);
        const int64_t spread = mask_id == CHILL_MASK_FULL ? cdiv(heads * items, slots) * one : heads * work / slots;
        const int64_t time = spread > one ? spread : one;
        if (k == 1 || time < best_time) {
            // (the first time is raised to it: an eighth has to be saved)
            best_time = k == 1 ? time * 7 / 8 : time;
            best = k;
        }
    }
    if (best == 1) return 0;
    const int most = cdiv(longest, best);
    // items sorted by their length, longest first, the parts of a q-tile next to each other
    constexpr int kMostKeyTiles = kFwdSplitMaxQTiles * 256 / 64;  // (q-tiles of at most 256 rows)
    int place[kMostKeyTiles + 1] = {};
    auto parts_of = [&](int i) { return tiles[i] > most ? cdiv(tiles[i], most) : 1; };
    auto length_of = [&](int i) { return cdiv(tiles[i], parts_of(i)); };
    for (int i = 0; i < n_q_tiles; i++) place[length_of(i)] += parts_of(i);
    int n_items = 0, partials = 0;
    for (int n = most; n >= 0; n--) {
        const int count = place[n];
        place[n] = n_items;
        n_items += count;
    }
    out->n_q_tiles = n_q_tiles;
    for (int i = n_q_tiles - 1; i >= 0; i--) {
        const int parts = parts_of(i);
        int& at = place[length_of(i)];
        for (int j = 0; j < parts; j++) out->item[at++] = i | j << 10 | parts << 15 | partials << 20;
        out->merge[i] = out->item[at - 1];
        if (parts > 1) partials += parts;
    }
    out->n_items = n_items;
    out->partials_per_head = partials;
    out->partial_floats = cfg.rows * D + 2 * cfg.waves * 64;  // O^T; m0 and l of every lane
    out->partials = static_cast<float*>(workspace);
    const int64_t partial_bytes = heads * partials * out->partial_floats * 4;
    out->again = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + partial_bytes);
    return partial_bytes + heads * n_q_tiles * 4;
}

}  // namespace chill
