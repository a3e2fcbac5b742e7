// Static MI355X tile table: (mask id, head dim, dtype, pass) -> tile shape.  It replaces the
// reference's per-GPU default tables and Triton autotune spaces (chill_attention/autotune.py:11-119,
// 129-240).  The functions are constexpr so the kernel launchers instantiate exactly the shapes the
// table reports through chill_tile_config().
//
// rows     = resident rows per workgroup (32 per wave): query rows in the forward and dQ passes,
//            key rows in the dK/dV pass;
// streamed = rows of one streamed LDS tile: keys in forward / dQ, queries in dK/dV.
#pragma once

#include "chill_params.h"

// Build-time overrides for the tile sweep (chill_attention/tune.py builds one library per candidate
// shape): 16-bit inputs with head dim <= 128 only.  Without them the table below is what ships.
#ifndef CHILL_TUNE_FWD_WAVES
#define CHILL_TUNE_FWD_WAVES 0
#endif
#ifndef CHILL_TUNE_FWD_STREAMED
#define CHILL_TUNE_FWD_STREAMED 0
#endif
#ifndef CHILL_TUNE_FWD_SMALL
#define CHILL_TUNE_FWD_SMALL 1
#endif
#ifndef CHILL_TUNE_FWD_STAGES
#define CHILL_TUNE_FWD_STAGES 0
#endif
#ifndef CHILL_TUNE_DQ_STAGES
#define CHILL_TUNE_DQ_STAGES 0
#endif
#ifndef CHILL_TUNE_DQ_WAVES
#define CHILL_TUNE_DQ_WAVES 0
#endif
#ifndef CHILL_TUNE_DQ_STREAMED
#define CHILL_TUNE_DQ_STREAMED 0
#endif
#ifndef CHILL_TUNE_DKDV_WAVES
#define CHILL_TUNE_DKDV_WAVES 0
#endif

// 1: the 8-wave forward of 16-bit inputs at head dim 128 streams 64-key tiles through four stages,
// the shape fwd_q_tile_fast and its generated loop are written for; 0: the shape before it (128-key
// tiles, two stages, fwd_q_tile).
#ifndef CHILL_FWD_FAST
#define CHILL_FWD_FAST 1
#endif

namespace chill {

constexpr int elem_bytes(int dtype) { return dtype == CHILL_F32 ? 4 : 2; }

// Forward LDS stage: a K tile padded for row-wise reads and a V tile padded for transposed reads
// (pads as in PaddedTile, chill_device.h).
constexpr int fwd_stage_bytes(int streamed, int D, int dtype) {
    const int rb = D * elem_bytes(dtype);
    const int vpad = dtype == CHILL_F32 ? 32 : (rb >= 128 ? 64 : 0);
    return streamed * (rb + 16) + streamed * (rb + vpad);
}

// Masks whose rows see a narrow band of keys: a q-tile is a short loop, and the time a workgroup
// spends before and after it (loading Q and the first K/V tile, storing O) is a large part of its
// life.  They get workgroups of four waves with a two-stage ring, two of which share a CU, so that one
// computes while the other loads or stores (measured: sliding window forward -22 %, dQ -16 %;
// chunkwise forward -5 %, dQ -14 %; on the causal workload the same shape re-reads K and V twice as
// often and is 1-2 % slower).
constexpr bool mask_is_banded(int mask_id) {
    return mask_id == CHILL_MASK_SLIDING_WINDOW || mask_id == CHILL_MASK_CHUNKWISE;
}
// The most keys a row of such a mask sees (`a0`, `a1` = the mask's first two arguments: left and right context, or
// chunk size and chunks looked back at); kWholeSequence for the other masks.  A wide band is a long loop again:
// the forward and dK/dV then take the shapes of the masks that are not banded, from the widths named at
// fwd_takes_short_row and dkdv_regs_serves_band on.
constexpr long long kWholeSequence = 1ll << 40;
constexpr long long mask_band_keys(int mask_id, long long a0, long long a1) {
    return mask_id == CHILL_MASK_SLIDING_WINDOW ? a0 + a1 + 1 : mask_id == CHILL_MASK_CHUNKWISE ? a0 * (a1 + 1) : kWholeSequence;
}
// (a banded mask of which only the id is known is taken to be narrow)
constexpr long long kNarrowBand = 1;

// Sequence lengths up to which the 4-wave shape also wins at head dim 128 for masks that are not banded
// (measured on causal and full masks, B8 H4 .. H16: forward -16 % at T = 512 and 1024, +20 % at 2085;
// dQ -24 % at 512, -14 % at 2048 and 4042, -5 % at 4096, +-1 % at 8192, where its extra K / V reads cost
// the neighbouring kernels more than it gains).  T = kLongSequence selects the long-sequence row.
constexpr int kLongSequence = 0x7fffffff;
constexpr int kFwdShortSequence = 1024;
constexpr int kFwdShortSequenceFull = 768;
constexpr int kDqShortSequence = 4096;
// The same shape is taken when the 8-wave one would leave CUs without a workgroup (B1 H8 T8192 causal:
// forward -7 %, dQ -17 %; with twice as many heads the 8-wave shape wins again).
constexpr int kComputeUnits = 256;
// (forward: only dQ still takes it; the 8-wave forward with its generated loop is 23 % faster than the 4-wave
// one at B1 H8 T8192)
// Banded masks take it while a row sees fewer than kFwdWideBand keys (measured at head dim 128, T = 8192 and 16384,
// the 8-wave shape against this one: sliding windows of 512 / 1024 / 2048 / 4096 keys +9 / -12 / -18 / -18 %,
// chunkwise 1024 x 2 -17 %, 128 x 3 +2 %).
constexpr int kFwdWideBand = 1024;
constexpr bool fwd_takes_short_row(int mask_id, long long band_keys, long long batch_heads, int T) {
    (void)batch_heads;
    // (under a full mask the 8-wave shape, whose loop is predicate-free from its first tile on, wins from 769 keys on:
    // B16 H16 T = 1024 / 1000 -12 / -7 %, T = 768 / 512 +2 / -1 %; causal T = 1024 / 768 / 512 +3 / +41 / +23 %)
    return T <= (mask_id == CHILL_MASK_FULL ? kFwdShortSequenceFull : kFwdShortSequence) ||
           (mask_is_banded(mask_id) && band_keys < kFwdWideBand);
}
constexpr bool dq_takes_short_row(long long batch_heads, int T) {
    return T <= kDqShortSequence || batch_heads * ((T + 255) / 256) <= kComputeUnits;
}

// Forward.  16-bit inputs at head dim 128: 8 waves (256 query rows), streamed tiles of 128 keys (half
// the barriers per key); narrow bands (fwd_takes_short_row), head dims <= 64 and short sequences: 4 waves, 64 keys, 2
// stages, two or three workgroups per CU (prefix-LM at D = 64: forward -14 %; causal at D = 16 .. 64:
// -5 .. -8 %).
constexpr int fwd_waves(int mask_id, int D, int dtype, int T) {
    if (dtype == CHILL_F32 || D > 128) return 4;
    if (CHILL_TUNE_FWD_WAVES) return CHILL_TUNE_FWD_WAVES;
    (void)mask_id;
    return (D <= 64 || T <= kFwdShortSequence) ? 4 : 8;
}
constexpr int fwd_streamed(int mask_id, int D, int dtype, int T) {
    if (dtype == CHILL_F32) return 32;
    if (D > 128) return 64;
    if (CHILL_TUNE_FWD_STREAMED) return CHILL_TUNE_FWD_STREAMED;
    return (fwd_waves(mask_id, D, dtype, T) == 8 && !CHILL_FWD_FAST) ? 128 : 64;
}
// LDS stages of the forward K/V ring: two for the 4-wave shape of 16-bit inputs (so that two
// workgroups fit a CU); otherwise three (one tile resident ahead, one in flight) when they fit in
// 144 KiB, else two.
constexpr int fwd_stages(int mask_id, int D, int dtype, int T) {
    const int streamed = fwd_streamed(mask_id, D, dtype, T);
    if (dtype != CHILL_F32 && D <= 128) {
        if (CHILL_TUNE_FWD_STAGES) return CHILL_TUNE_FWD_STAGES;
        // the fast forward keeps one tile resident ahead of the one in use: three stages (two workgroups of
        // four waves still share a CU at head dim 64), four for the 8-wave workgroup that owns its CU
        if (fwd_waves(mask_id, D, dtype, T) == 4) return (CHILL_FWD_FAST && D == 64) ? 3 : 2;
        if (CHILL_FWD_FAST) return 4;
    }
    return 3 * fwd_stage_bytes(streamed, D, dtype) <= 144 * 1024 ? 3 : 2;
}
// 16-bit inputs at head dim 256: fwd_regs_kernel (O^T in hand-managed accumulation registers).
constexpr bool fwd_uses_regs(int D, int dtype) { return dtype != CHILL_F32 && D == 256; }

// Forward launches far too small for the chip (fwd_small_kernel): a workgroup of four waves owns 32
// query rows and its waves split the keys.  Per wave LDS holds a 32-row K block, a 32-row V block and
// the wave's running max and row sum; rows of at most 512 bytes, so that four such areas fit.
// For 16-bit inputs it is taken while its grid of B * H * T / 32 tiles is about what the chip holds at once
// (measured against the ordinary forward, causal and full masks, T = 128 .. 16384, 1 .. 128 heads: with up to
// 256 tiles it wins everywhere, by 1.1x .. 1.5x; with 512 it still wins at head dim 128, where a block is more
// work, and under causal-like masks; with 1024 it loses or ties); fp32 much further up (fwd_small_max_tiles).
constexpr int kFwdSmallWaves = 4;
// (sequences of up to 16384 rows: with a head or two of such a sequence the ordinary kernels have a few dozen workgroups.
// Measured at T = 8192: fp32 causal B1 H2 D64 forward 633 -> 193 us, dQ 883 -> 244, dK/dV 1032 -> 332, full mask
// 645 -> 340, 908 -> 408, 1047 -> 597; fp32 causal B1 H4 T16384 forward 1318 -> 1224, dQ 2800 -> 1570; bf16 causal
// B1 H2 D128 forward 142 -> 89, dQ 153 -> 90, full mask 145 -> 125 and 156 -> 132; bf16 causal B1 H1 D64 dQ 108 -> 54,
// dK/dV 110 -> 76)
constexpr int kFwdSmallMaxT = 16384;
// (at the end the area also takes the wave's partial O^T, 4 KiB per 32 columns of the head dim)
// (fp32 at head dims up to 128 has kernels of the same shape whose products go through bf16 parts, chill_f32_parts.h: their
// areas hold the parts of one 32-row block of V, in dQ of K, which are smaller, in dK/dV, at head dims up to 64, of Q and of dO)
constexpr bool f32_parts_serve(int D, int dtype) { return dtype == CHILL_F32 && D <= 128; }
constexpr int f32_planes_bytes(int D) { return 3 * 32 * D * 2; }
constexpr int fwd_small_wave_bytes(int D, int dtype) {
    const int blocks = 2 * 32 * D * elem_bytes(dtype), partial = ((D + 31) / 32) * 16 * 64 * 4;
    return (blocks > partial ? blocks : partial) + 2 * 64 * 4;
}
constexpr int fwd_small_lds_bytes(int D, int dtype) { return kFwdSmallWaves * fwd_small_wave_bytes(D, dtype); }
// fp32, whose ordinary kernels give a wave 32 rows and all their keys at 2 us and more per block, is served much
// further up since the small kernels balance their launches (small_takes_two_tiles, below).  Measured against
// fwd_kernel / dq_kernel / dkdv_kernel at head dims 32, 64 and 128, T = 512 .. 4096, 1536 .. 32768 tiles: under
// masks whose rows grow with their index (causal, prefix-LM) the forward wins up to 2048 tiles (B1 H24 T2048 D64:
// 300 -> 154 us; at 2048 tiles 373 -> 359, at 4096 +5 .. +9 %; head dim 128: 387 -> 317 at 1536 tiles, +11 .. +15 %
// at 2048), dQ up to 16384 tiles (8192 at head dim 128; B1 H24 T2048: 406 -> 195 us; B4 H16 T4096: 2000 -> 1750; head dim 128: 3925 -> 3820),
// dK/dV up to 4096 tiles at T <= 2048 (B4 H16 T2048: 797 -> 715 us; prefix-LM B8 H32 T1024, 8192 tiles: +9 %) and 1024
// at T = 4096 (B1 H8: 523 -> 333 us; B1 H16: 606 -> 645); under the other masks, whose tiles are all alike, forward
// and dQ win up to 1536 tiles (full mask B1 H24 T2048 D64: 318 -> 276 and 421 -> 337 us; sliding window 70 -> 60 and
// 104 -> 85) and tie or lose from 2048 on, and dK/dV does not win beyond its 512.
constexpr bool mask_rows_grow(int mask_id) { return mask_id == CHILL_MASK_CAUSAL || mask_id == CHILL_MASK_PREFIX_LM; }
constexpr long long fwd_small_max_tiles(int mask_id, int D, int dtype) {
    // (16-bit head dims <= 64 at 512 tiles: causal B1 H2 T8192 69 -> 57 us, B1 H4 T4096 38 -> 31; full mask 71 -> 81, 39 -> 42)
    if (dtype != CHILL_F32) return ((D >= 128 || mask_rows_grow(mask_id)) ? 2 : 1) * kComputeUnits;
    return (mask_rows_grow(mask_id) && D <= 64 ? 8 : 6) * kComputeUnits;
}
constexpr bool fwd_takes_small(int mask_id, long long batch_heads, int T, int D, int dtype) {
    return CHILL_TUNE_FWD_SMALL && D * elem_bytes(dtype) <= 512 && T <= kFwdSmallMaxT &&
           batch_heads * ((T + 31) / 32) <= fwd_small_max_tiles(mask_id, D, dtype);
}

// With more 32-row tiles than the chip has CUs the workgroups of a launch no longer run all at once or alone on their
// CUs, and under causal-like masks, where a tile's work grows with its index, the launch ends when the CU with the
// longest tiles does.  Then, in the forward and dQ, a workgroup of eight waves takes two tiles side by side, tile j
// from the end and tile j from the start of a head, which add up to the same work for every workgroup, where two areas
// fit in LDS (the wave then has 256 registers: enough for the forward and dQ, not for dK/dV with K, V and two
// accumulators); and every small launch takes its tiles longest first across all heads.  Measured on fp32 at head dim
// 64, forward / dQ / dK/dV: prefix-LM B1 H8 T2048 83 / 127 / 161 -> 66 / 87 / 127 us, causal 81 / 126 / 159 ->
// 52 / 69 / 97, causal B2 H8 T1024 45 / 71 / 90 -> 30 / 40 / 58; two tiles per workgroup against the new order
// alone: forward 66 against 69, dQ 87 against 101 us on the prefix-LM shape.
constexpr bool small_fits_two_tiles(int lds_bytes_one) { return 2 * lds_bytes_one <= 160 * 1024; }
constexpr bool small_takes_two_tiles(long long tiles) { return tiles > kComputeUnits; }
// With no more tiles than CUs a workgroup has its CU to itself, and two sets of four waves share the streamed blocks of its tile
// where a row reaches over enough of them to pay for the longer merge.  us, one set -> two, bf16
// causal where not named: forward D64 B1 H8 T256 5.7 -> 5.9, T512 7.7 -> 7.0, T1024 11.2 -> 9.1, fp16 H4 T300 7.2 -> 6.3, full mask
// H2 T2048 17.2 -> 12.7, window 64 H4 T1024 5.4 -> 5.6, D128 H4 T512 9.7 -> 9.2, T2048 24.0 -> 17.2, prefix-LM H1 T8192 86 -> 48;
// dK/dV D64 H8 T160 7.7 -> 7.4, T512 9.9 -> 8.8, T1024 14.6 -> 11.2, window 64 7.4 -> 7.8, prefix-LM H1 T8192 78 -> 45; dQ D64 H8 T512
// 8.5 -> 8.8, T1024 11.5 -> 10.5, D128 H4 T512 12.7 -> 13.9, B2 H4 T800 16.2 -> 15.3, T2048 25.8 -> 21.5, prefix-LM H1 T8192 85 -> 54,
// window 32 of T3000 9.6 -> 11.1.  fp32, the forward alone (graph replay, causal D64 where not named): B1 H2 T256 9.78 -> 9.83,
// B2 H8 T384 12.97 -> 12.16, T512 15.28 -> 14.15, B1 H4 T1111 29.2 -> 24.4, H8 T1024 25.2 -> 22.4, H1 T8192 175 -> 139, full mask T256 10.05 -> 9.87, window
// 32 + 0 T1024 7.74 -> 8.45, 64 + 64 10.87 -> 10.28, 128 + 128 13.65 -> 12.75.
constexpr bool small_takes_two_sets(int mask_id, int dtype, int pass, long long tiles, int T, long long band_keys) {
    const long long reach = T < band_keys ? T : band_keys;
    if (tiles > kComputeUnits) return false;
    if (dtype == CHILL_F32) return pass == CHILL_PASS_FWD && reach > (mask_rows_grow(mask_id) ? 256 : 128);
    return reach > (pass == CHILL_PASS_FWD ? 256 : pass == CHILL_PASS_DQ ? 768 : 128);
}
// what the report says of a small launch: 32 rows and the waves of a tile, four or, in two sets, eight; the LDS of the workgroup,
// which takes two tiles of four waves or one tile with two sets
constexpr TileConfig small_tile_config(int mask_id, int dtype, int pass, int lds_bytes_one, long long tiles, int T, long long band_keys) {
    const bool fits = small_fits_two_tiles(lds_bytes_one);
    const bool two = fits && pass != CHILL_PASS_DKDV && small_takes_two_tiles(tiles);
    const bool sets = fits && small_takes_two_sets(mask_id, dtype, pass, tiles, T, band_keys);
    return TileConfig{32, 32, sets ? 2 * kFwdSmallWaves : kFwdSmallWaves, two || sets ? 2 * lds_bytes_one : lds_bytes_one};
}

// The backward of such launches (dq_small_kernel, dkdv_small_kernel): the same split of the streamed
// axis over four waves; a wave's area holds two 32-row blocks (K and V, or Q and dO), later its partial
// accumulators (`outputs` x 4 KiB per 32 columns of the head dim), and LSE2 / delta of a query block.
#ifndef CHILL_TUNE_BWD_SMALL
#define CHILL_TUNE_BWD_SMALL 1
#endif
// (`in_parts`: dK/dV of fp32 through bf16 parts holds three planes of both, half as much again)
constexpr int bwd_small_wave_bytes(int D, int dtype, int outputs, bool in_parts = false) {
    const int rows = 2 * 32 * D * elem_bytes(dtype), planes = in_parts ? outputs * f32_planes_bytes(D) : 0;
    const int blocks = rows > planes ? rows : planes, partial = outputs * ((D + 31) / 32) * 16 * 64 * 4;
    return (blocks > partial ? blocks : partial) + 2 * 32 * 4;
}
constexpr int bwd_small_lds_bytes(int D, int dtype, int outputs, bool in_parts = false) {
    return kFwdSmallWaves * bwd_small_wave_bytes(D, dtype, outputs, in_parts);
}
#ifndef CHILL_TUNE_BWD_SMALL_SCALE
#define CHILL_TUNE_BWD_SMALL_SCALE 1
#endif
// Where they win (measured against dq_kernel / dkdv_kernel on causal masks, 1 .. 128 heads, T = 128 .. 4096):
// dQ while its grid of B * H * T / 32 workgroups is at most 512 (256 for 16-bit inputs at head dim 128):
// 1.1x .. 1.9x for 16-bit inputs, 1.5x .. 3.8x for fp32; dK/dV at head dims up to 64 with at most 256 workgroups
// (512 for fp32): 1.1x .. 1.4x and 1.2x .. 3.4x.  At head dim 128 dK/dV does not win (a wave then holds K, V and
// two accumulators of 64 registers each), and fp32 rows of 512 bytes do not fit a wave's registers at all.
constexpr bool bwd_small_serves(int D, int dtype, int pass) {
    return CHILL_TUNE_BWD_SMALL && (pass == CHILL_PASS_DKDV ? D <= 64 : (D <= 128 && D * elem_bytes(dtype) <= 512));
}
// (fp32 beyond that: the measurements at fwd_small_max_tiles)
constexpr long long bwd_small_max_tiles(int mask_id, int T, int D, int dtype, int pass) {
    // (16-bit dQ at 512 tiles, head dim 128: causal B1 H2 T8192 153 -> 90 us, B1 H4 T4096 82 -> 50, B1 H16 T1024 27 -> 23, full
    // mask 156 -> 132 and 95 -> 75; at 1024 tiles wins and losses of up to 25 % either way)
    // (16-bit dK/dV at 512 tiles, head dim 64, causal: B1 H2 T8192 118 -> 90 us, B1 H4 T4096 62 -> 52, B1 H16 T1024 20 -> 22; full
    // mask 134 -> 164 and 76 -> 91)
    if (dtype != CHILL_F32) return ((pass == CHILL_PASS_DQ || (mask_rows_grow(mask_id) && T >= 4096)) ? 2 : 1) * kComputeUnits;
    // (dQ at 16384 tiles, causal B8 H16 T4096: head dim 64 3775 -> 3393 us, 32 2045 -> 1901, 128 7822 -> 7909; at 32768 +1 .. +14 %)
    if (pass == CHILL_PASS_DQ) return (mask_rows_grow(mask_id) ? (D <= 64 ? 64 : 32) : 6) * kComputeUnits;
    return (mask_rows_grow(mask_id) ? (T <= 2048 ? 16 : 4) : 2) * kComputeUnits;
}
constexpr bool bwd_takes_small(int mask_id, long long batch_heads, int T, int D, int dtype, int pass) {
    return bwd_small_serves(D, dtype, pass) && T <= kFwdSmallMaxT * CHILL_TUNE_BWD_SMALL_SCALE &&
           batch_heads * ((T + 31) / 32) <= bwd_small_max_tiles(mask_id, T, D, dtype, pass) * CHILL_TUNE_BWD_SMALL_SCALE;
}
// fp32 launches whose products go through bf16 parts: all at head dim 16; at head dims 32 and 64 those of more than 256 and of at least
// 1024 rows, bands of less than 256 keys aside, and those of more than 2048 tiles of key / value heads, which no pass leaves to the
// small kernels; at head dim 128 those of at least 1024 rows, or 512 with at most one tile a CU, bands of less than 512 keys aside, and
// those of at least 1024 tiles of query heads.  Below that a small forward ends before the splits of a wave's first operands are paid for, and the passes go
// together: P comes out of a score and an LSE2 of the same rounding (dQ of scores up to 50, B1 H8 T1024, off by 2.2e-6 with both
// through the fp32 instruction, 2.0e-6 with both through parts, 4.2e-6 with one of each).
// Forward / dQ / dK/dV in us, fp32 instruction -> parts, in the kernels of few tiles (chill_f32_fwd_small.h, chill_f32_bwd_small.h):
//   D64 causal B1 H8 T1024 22 / 31 / 41 -> 24 / 22 / 30   B1 H4 T1111 24 / 36 / 45 -> 25 / 23 / 32   B2 H16 T2048 166 / 231 / 337 -> 162 / 187 / 262
//       full mask B1 H8 T2048 78 / 104 / 144 -> 72 / 83 / 114   window 256 B1 H8 T2048 19 / 28 / 39 -> 20 / 23 / 34
//   D128 (dK/dV in the kernel of launches that fill the chip, which is ahead however few tiles there are: the parts of Q and dO of four
//        waves do not fit in LDS)   causal B1 H8 T512 23 / 35 / 164 -> 24 / 27 / 80   B1 H8 T1024 42 / 61 / 317 -> 41 / 44 / 148
//       B1 H24 T1024 77 / 115 / 319 -> 82 / 92 / 150   B1 H8 T2048 89 / 128 / 623 -> 89 / 98 / 282   B1 H2 T8192 341 / 474 / 2516 -> 330 / 361 / 1144
//       full mask B1 H8 T2048 155 / 216 / 628 -> 152 / 168 / 290   window 256 + 256 B1 H4 T2048 30 / 43 / 201 -> 30 / 34 / 98
//   D32 causal B1 H8 T512 9 / 11 / 14 -> 10 / 9 / 12   B1 H16 T1100 28 / 41 / 34 -> 28 / 31 / 27   D16 B8 H8 T256 6.5 / 7.1 / 9.1 -> 5.8 / 6.1 / 7.8
//       B4 H8 T1100 32 / 36 / 43 -> 25 / 29 / 32
//   outside the rule, the forward alone: D64 causal B2 H16 T512 18 -> 20   window 100 + 30 B1 H4 T1111 10 -> 12   D128 causal B1 H8 T256 15.9 -> 18.3
//       B4 H8 T512 37.1 -> 38.7   window 100 + 30 B1 H16 T1024 34.2 -> 37.8   chunkwise 128, 2 B1 H8 T4001 85.4 -> 90.4
// and in those that fill the chip (chill_f32_group.h):
//   D64 causal B4 H16 T4096 1119 / 1708 / 2209 -> 745 / 971 / 1531   B8 H32 T300 55 / 96 / 139 -> 38 / 47 / 72   B32 H32 T128 49 / 118 / 163 -> 39 / 50 / 86
//       full mask B4 H16 T4096 2101 / 3014 / 4227 -> 1428 / 1885 / 2822   window 100 + 30 B8 H32 T800 182 / 207 / 329 -> 94 / 125 / 205
//   D32 causal B4 H16 T4096 660 / 987 / 1147 -> 409 / 539 / 758   D16 503 / 592 / 920 -> 350 / 403 / 660
//   D128 causal B4 H16 T4096 2300 / 3605 / 5325 -> 1708 / 2175 / 2865   B1 H32 T2048 301 / 495 / 695 -> 220 / 278 / 372   B8 H32 T300 123 / 219 / 213 -> 90 / 118 / 133
//       window 100 + 30 B8 H32 T800 440 / 482 / 660 -> 232 / 307 / 368   16 + 16 B8 H8 T3000 258 / 333 / 442 -> 165 / 224 / 275
//       grouped heads B4 H32/8 T2085 1493 / 2043 / 3044 -> 972 / 1277 / 1666   B4 H32/4 T512 109 / 209 / 1253 -> 83 / 107 / 566
//   D128 of 1024 tiles: causal B1 H16 T2048 169 / 248 / 628 -> 179 / 218 / 289   B1 H4 T8192 610 / 855 / 2522 -> 688 / 832 / 1119   B8 H32 T128 41 / 69 / 54 -> 23 / 31 / 38
//       full mask B1 H16 T2048 327 / 441 / 643 -> 198 / 260 / 355
// (Counting key / value heads at head dims 32 and 64 keeps grouped launches on the fp32 instruction that would be faster through parts in
// all passes, by the query heads: window 100 + 30 B8 H32/8 T800 D64 181 / 203 / 355 -> 93 / 116 / 197, causal 235 / 374 / 397 -> 147 /
// 191 / 312, T300 56 / 97 / 84 -> 36 / 45 / 67.  That is not done yet.)
constexpr long long f32_group_tiles(int D) { return D == 128 ? 4 * kComputeUnits - 1 : 8 * kComputeUnits; }
constexpr bool f32_takes_group(long long heads, int T, int D) { return heads * (((long long)T + 31) / 32) > f32_group_tiles(D); }
constexpr bool f32_all_parts(int D, int dtype) { return f32_parts_serve(D, dtype) && D < 32; }
constexpr bool f32_takes_parts(long long band_keys, long long heads, long long kv_heads, int T, int D, int dtype) {
    if (!f32_parts_serve(D, dtype)) return false;
    if (f32_all_parts(D, dtype) || f32_takes_group(D == 128 ? heads : kv_heads, T, D)) return true;
    if (D == 128) return band_keys >= 512 && (T >= 1024 || (T >= 512 && heads * ((T + 31) / 32) <= kComputeUnits));
    return band_keys >= 256 && T >= (D == 32 ? 257 : 1024);
}
// A forward without LSE2 has no backward that must see its rounding.  On few tiles at head dims 32 and 64 it takes the parts only where
// they are ahead by themselves; the two report the same workgroup.  us, fp32 instruction -> parts:
//   D32 causal B1 H8 T384 7.3 -> 8.4   T512 8.8 -> 9.5   full mask H8 T384 7.4 -> 8.5   window 255 + 1 H16 T2048 19.8 -> 21.9, H40 T1024 25.2 -> 29.3   chunkwise 128, 2
//       H12 T2048 18.6 -> 21.2;   causal B1 H8 T1000 14.7 -> 13.3   H14 T1100 20.0 -> 16.3   B2 H16 T1024 25.4 -> 27.3   B2 H24 T1024 47.2 -> 40.2   B2 H16
//       T1500 63.2 -> 50.5   window 1023 + 0 H12 T4096 69.1 -> 62.2
//   D64 causal B1 H2 T1024 21.6 -> 22.9   window 255 + 1 H2 T2048 11.3 -> 13.9, 511 + 0 H2 T4096 15.8 -> 17.2;   causal B1 H8 T1100 29.1 -> 26.3   H24 T1300
//       59.2 -> 56.4   H12 T3000 167 -> 152   window 1023 + 0 H12 T4096 122 -> 113
constexpr bool f32_forward_alone_takes_parts(long long band_keys, int T, int D) {
    return (D != 32 && D != 64) || (band_keys >= 1024 && T >= (D == 32 ? 1000 : 1025));
}
// The kernels of launches that fill the chip: 128 rows a workgroup, two stages of the parts of 32 rows of K and V, in dK/dV of Q and
// dO with LSE2 and delta.  They take every launch that the small kernels do not, of those launches the dQ and dK/dV of more than
// 2048 tiles too (causal D64, dQ B4 H16 T4096 1338 -> 971 us, B4 H16 T2048 394 -> 263; dK/dV 498 -> 415; at 2048 tiles 197 -> 143 and
// 251 -> 199, at 1024 103 -> 116 and 129 -> 166), and at head dim 128 all of at least 1024.
// (dQ at head dim 64: the low parts of dO, a thread's 16 bytes of each of four operands)
constexpr bool f32_group_parks(int D) { return D == 64; }
constexpr TileConfig f32_group_tile_config(int D, int pass) {
    const int stage = 2 * f32_planes_bytes(D) + (pass == CHILL_PASS_DKDV ? 2 * 32 * 4 : 0);
    return TileConfig{128, 32, 4, 2 * stage + (pass == CHILL_PASS_DQ && f32_group_parks(D) ? 4 * 64 * 16 * (D / 16) : 0)};
}
// Workgroups that share a CU (work_item's `resident`), by the kernels' registers and LDS.  (Forward and dQ at head dim 128 with 2, by
// which the second half of a grid of 257 to 512 came shortest first: causal B1 H32 T2048 259 / 331 us where longest first takes 216 / 278,
// H16 T4096 486 / 627 and 407 / 532; the forward at head dims 32 and 16 with 2: B2 H24 T2048 99 and 87 us, 90 and 78 with 4; dQ at 16 92, 84)
constexpr int f32_group_resident(int D, int pass) {
    if (D == 128) return 1;
    if (pass == CHILL_PASS_DKDV) return D == 64 ? 1 : 2;
    return D == 64 ? 2 : pass == CHILL_PASS_FWD ? 4 : D == 32 ? 2 : 3;
}
constexpr bool f32_group_resident_fits(int D) {
    return f32_group_resident(D, CHILL_PASS_FWD) * f32_group_tile_config(D, CHILL_PASS_FWD).lds_bytes <= 160 * 1024 &&
           f32_group_resident(D, CHILL_PASS_DQ) * f32_group_tile_config(D, CHILL_PASS_DQ).lds_bytes <= 160 * 1024 &&
           f32_group_resident(D, CHILL_PASS_DKDV) * f32_group_tile_config(D, CHILL_PASS_DKDV).lds_bytes <= 160 * 1024;
}
static_assert(f32_group_resident_fits(16) && f32_group_resident_fits(32) && f32_group_resident_fits(64) && f32_group_resident_fits(128), "LDS");
constexpr TileConfig fwd_tile_config(int mask_id, int D, int dtype, int T = kLongSequence) {
    const int waves = fwd_waves(mask_id, D, dtype, T);
    const int streamed = fwd_streamed(mask_id, D, dtype, T);
    return TileConfig{waves * 32, streamed, waves,
                      fwd_stages(mask_id, D, dtype, T) * fwd_stage_bytes(streamed, D, dtype)};
}

// dQ.  16-bit inputs at head dim 128: 8 waves x 64 streamed keys in three stages; banded masks, head
// dims <= 64 and sequences up to kDqShortSequence: 4 waves x 64 keys in two stages, two workgroups per
// CU (prefix-LM at D = 64: dQ -9 %).  16-bit inputs at head dim 256: dq_regs_kernel (hand-managed
// accumulation registers), 4 waves, dq_regs_keys streamed keys per tile (0: the shape is served by
// dq_kernel).
constexpr int dq_regs_keys(int D, int dtype) { return (dtype != CHILL_F32 && D == 256) ? 32 : 0; }
constexpr int dq_waves(int mask_id, int D, int dtype, int T) {
    if (dtype == CHILL_F32 || D > 128) return 4;
    if (CHILL_TUNE_DQ_WAVES) return CHILL_TUNE_DQ_WAVES;
    return (mask_is_banded(mask_id) || D <= 64 || T <= kDqShortSequence) ? 4 : 8;
}
constexpr int dq_streamed(int D, int dtype) {
    if (dtype == CHILL_F32) return 32;
    if (D > 128) return dq_regs_keys(D, dtype) > 0 ? dq_regs_keys(D, dtype) : 32;
    return CHILL_TUNE_DQ_STREAMED ? CHILL_TUNE_DQ_STREAMED : 64;
}
// dQ LDS stage: swizzled (unpadded) K and V tiles.  Two stages for the 4-wave shape of 16-bit inputs;
// otherwise three when they fit in 144 KiB.
constexpr int dq_stages(int mask_id, int D, int dtype, int T) {
    if (dtype != CHILL_F32 && D <= 128) {
        if (CHILL_TUNE_DQ_STAGES) return CHILL_TUNE_DQ_STAGES;
        if (dq_waves(mask_id, D, dtype, T) == 4) return 2;
    }
    return 3 * 2 * dq_streamed(D, dtype) * D * elem_bytes(dtype) <= 144 * 1024 ? 3 : 2;
}

// 16-bit inputs at head dim 128 have a second dQ kernel (dq_regs2_kernel): 4 waves, one per SIMD, 64 query rows each
// with Q and dO in registers, 32-key tiles in four stages, runs of predicate-free tiles in a generated loop
// (gen_dq_loop.py).  It owns its CU; taken like its dK/dV counterpart for long sequences on grids of at least two
// workgroups per CU, not for the banded masks.  Measured on dQ alone, against dq_kernel on one box: causal B8 H16
// T8192 2.71 / 2.90 ms, B2 H8 T8192 0.408 / 0.428, prefix-LM B4 H16 T8192 1.45 / 1.55, full mask fp16 B4 H16 T4096
// 0.76 / 0.82; but causal B16 H16 T4096 1.63 / 1.62, B8 H8 T4096 0.509 / 0.496, B1 H8 T8192 0.227 / 0.232.
// (from 4097 keys on, where dq_kernel leaves its 4-wave shape; full masks from 2048.  Measured on bf16 at B8 H16 since
// the waves at a ragged end of the sequence take the complete tile's predicate-free range: causal T = 5000 / 6143 /
// 7000 / 8000 -7.7 / -8.1 / -4.9 / -5.3 %, at T = 4096 / 3072 / 2048 against the 4-wave shape +2 / +3 / +14 %; full mask
// T = 2048 / 3072 / 4096 / 6143 / 8000 -4 / -7 / -7 / -9.5 / -9.6 %; prefix-LM T = 5000 / 7000 -6.4 %, T = 3072 +0.5 %)
constexpr int dq_regs2_min_sequence(int mask_id) { return mask_id == CHILL_MASK_FULL ? 2048 : 4097; }
constexpr int kDqRegs2MinWorkgroups = 2 * 256;
constexpr bool dq_regs2_is_optional(int D, int dtype) { return dtype != CHILL_F32 && D == 128; }
constexpr bool dq_takes_regs2(int mask_id, long long batch_heads, int T) {
    return !mask_is_banded(mask_id) && T >= dq_regs2_min_sequence(mask_id) && batch_heads * ((T + 255) / 256) >= kDqRegs2MinWorkgroups;
}
constexpr TileConfig dq_regs2_tile_config(int D, int dtype) {
    return TileConfig{256, 32, 4, 4 * 2 * 32 * D * elem_bytes(dtype)};
}

// fp32 at head dim 256 (dq_split_kernel): two waves share a 32-query block; two stages of 32-key K and V
// tiles, then one 4 KiB slot per wave for the two products of a block.
constexpr bool dq_is_split(int D, int dtype) { return dtype == CHILL_F32 && D == 256; }
constexpr TileConfig dq_tile_config(int mask_id, int D, int dtype, int T = kLongSequence) {
    const int waves = dq_waves(mask_id, D, dtype, T);
    const int streamed = dq_streamed(D, dtype);
    if (dq_is_split(D, dtype)) return TileConfig{waves * 16, 32, waves, 2 * 2 * 32 * D * 4 + waves * 16 * 64 * 4};
    return TileConfig{waves * 32, streamed, waves,
                      dq_stages(mask_id, D, dtype, T) * 2 * streamed * D * elem_bytes(dtype)};
}

// dK/dV, rows of at most 256 bytes ("paired" kernel): a workgroup of 8 waves owns 128 key rows;
// pairs of waves share a 32-key block and split the streamed 64-row query tiles.  LDS: the resident
// K and V tiles plus two ring stages of swizzled Q and dO tiles with the LSE2 and delta of their rows.
// Longer rows: dkdv_split_kernel, below.
constexpr bool dkdv_is_paired(int D, int dtype) { return D * elem_bytes(dtype) <= 256; }
// 16-bit head dims <= 64: workgroups of 4 waves (64 key rows), small enough in LDS (50 KiB at D = 64)
// and registers (167) for two or three of them per CU, which hide each other's start and end
// (measured: sliding window dK/dV -32 %, prefix-LM at D = 64 -17 %).  At D = 128 the two-stage ring of
// such a workgroup takes 99 KiB; with a one-stage ring it fits twice (dkdv_takes_one_stage).
// `small_grid`: the 8-wave grid would cover at most half of the CUs, or not all of them under a mask whose rows grow with their
// index, where one round of 8-wave workgroups lasts as long as the longest of them (dkdv_takes_small_row); then the
// 64-row workgroup is taken at every 16-bit head dim.  D128 bf16, 8-wave workgroups, us, 8 waves -> 4: 128 causal B1 H8 T2048 -17 %; 160
// 61 -> 49; 192 B2 H32/4 T3000 510 -> 406; 224 B1 H8 T3500 83 -> 66, prefix-LM 88 -> 75, full mask 20 workgroups a head, 160, 62 -> 91,
// window 512 24 -> 32; 288 B1 H9 T4000 99 -> 100; 320 B2 H32/8 T2500 249 -> 269.  (From 256 on dkdv_takes_one_stage has those grids.)
constexpr int dkdv_paired_waves(int mask_id, int D, int dtype, bool small_grid = false) {
    (void)mask_id;
    if (CHILL_TUNE_DKDV_WAVES) return CHILL_TUNE_DKDV_WAVES;
    return (dtype != CHILL_F32 && (D <= 64 || small_grid)) ? 4 : 8;
}
constexpr bool dkdv_takes_small_row(int mask_id, long long batch_kv_heads, int T) {
    return batch_kv_heads * ((T + 127) / 128) <= (mask_rows_grow(mask_id) ? kComputeUnits - 1 : kComputeUnits / 2);
}
// Narrow bands at head dim 128, 16-bit: the 64-row workgroup with a ring of ONE stage (64.5 KiB), two of which share a CU.  Its
// loads are exposed, but a key block of a band has a handful of query tiles, and what the 8-wave workgroup, alone on its CU, spends
// before and after them (K and V to LDS, the exchange of the pairs, the stores) hides behind the other workgroup.  us, 8 waves ->
// one stage: window 16 + 16 fp16 B8 H4 T6000 101 -> 79, bf16 B2 H16/4 T2085 36 -> 27; 128 + 128 115 -> 95, 44 -> 33, bf16 B2 H32
// T4096 153 -> 128; 512 + 128 172 -> 160, 75 -> 57; 1024 + 0 231 -> 219; 2047 + 0 352 -> 346, B2 H16/4 T16000 917 -> 905; 3000 + 500
// 523 -> 529; chunkwise 100 x 3 129 -> 113, 128 x 3 114 -> 105, B2 H16 T3000 55 -> 49, 1000 x 2 392 -> 385 (T3000 180 -> 183),
// 1000 x 5 640 -> 642 (T3000 192 -> 200).  Letting dO's half of the next tile go out behind the dV^T MFMAs, with a barrier of its own,
// costs 2-10 %.
// Under masks whose rows grow with their index the smaller workgroups end a launch more evenly, the more so over the unequal
// sequences of a padded batch.  Training step, us, 8 waves -> one stage (bf16; the number is that of 8-wave workgroups): causal 256
// B1 H16/4 T8192 1272 -> 1216, B4 H32/8 T1000 226 -> 210; 272 B2 H32/8 T2085 411 -> 388; 384 B1 H12 T4000 280 -> 274; 512 B1 H32 T2048
// 194 -> 195; 752 B2 H8 T6000 649 -> 644; 960 B4 H12 T2500 386 -> 384; 1536 B8 H16 T1500 424 -> 430; 2176 B8 H16 T2085 739 -> 737;
// prefix-LM 384 285 -> 272, 512 199 -> 196, 960 394 -> 385, 1536 434 -> 435; padded to T/4 .. T, causal B8 H16 T300 56 -> 50, B4 H32/8
// T2085 479 -> 463, B8 H16 T1500 285 -> 273, T2085 448 -> 435, B4 H32 T2900 817 -> 823, prefix-LM 344 -> 317, 297 -> 284, 463 -> 450,
// 835 -> 831.  Full masks are within 1 % either way.
// Grids of fewer 8-wave workgroups than CUs keep the two-stage 64-row workgroups (dkdv_takes_small_row), those of at least as many
// leave them.  Around the line the loop of a workgroup decides, long ones for two stages; backward, us, two stages -> one, causal and
// prefix-LM: 192 B3 H16/4 T2048 222 -> 230, 219 -> 243; 224 B1 H8 T3500 133 -> 136, 132 -> 137; 240 B1 H16 T1900 87 -> 84, 92 -> 85;
// 248 B1 H8 T3968 154 -> 157, 157 -> 158; 255 B1 H17 T1900 91 -> 87, 96 -> 88; 256 B1 H16 T2048 91 -> 90, 96 -> 91, B2 H16/8 T2048
// 140 -> 141, 153 -> 145, B1 H16/4 T8192 914 -> 970, 913 -> 1002; 272 B1 H17 T2048 101 -> 96, 103 -> 99; 384 B1 H12 T4000 216 -> 190,
// 217 -> 193.
// (The report is that of a launch without lengths: a padded one takes these workgroups on larger grids too.)
constexpr int kDkdvOneStageBand = 2048;
constexpr int kDkdvOneStageMaxGrid = 4 * kComputeUnits;
constexpr bool dkdv_one_stage_serves(int mask_id, int D, int dtype) {
    return dtype != CHILL_F32 && D == 128 && (mask_is_banded(mask_id) || mask_rows_grow(mask_id));
}
constexpr bool dkdv_takes_one_stage(int mask_id, long long band_keys, long long batch_kv_heads, int T, bool padded) {
    return mask_is_banded(mask_id) ? band_keys <= kDkdvOneStageBand
                                   : padded || batch_kv_heads * ((T + 127) / 128) < kDkdvOneStageMaxGrid;
}
// at the end the waves of a pair exchange one fp32 accumulator each through LDS: 8 waves x (D rounded
// up to 32) x 32 floats
constexpr int dkdv_paired_exchange_bytes(int D) { return 8 * ((D + 31) / 32) * 16 * 64 * 4; }
// Longer rows (fp32 at head dims 128 and 256, dkdv_split_kernel): dkdv_split(D) waves share a 32-key
// block and its state; two ring stages of 32-row Q and dO tiles, then one 4 KiB slot per wave for the
// partial products.  Head dim 128: 8 waves, 128 key rows, two waves per SIMD; head dim 256: 4 waves
// on one 32-key block (two ring stages alone take 128 KiB).
constexpr int dkdv_split(int D) { return D >= 256 ? 4 : 2; }
constexpr int dkdv_split_waves(int D) { return D >= 256 ? 4 : 8; }
constexpr int dkdv_split_stage_bytes(int D, int dtype) { return 2 * 32 * D * elem_bytes(dtype) + 2 * 32 * 4; }
constexpr int dkdv_split_lds_bytes(int D, int dtype) {
    return 2 * dkdv_split_stage_bytes(D, dtype) + dkdv_split_waves(D) * 16 * 64 * 4;
}

// dK/dV with hand-managed accumulation registers (dkdv_regs_kernel, 16-bit inputs): 4 waves, K in
// registers, V in LDS, 32-row Q / dO tiles in a ring.  blocks = 32-key blocks per wave:
//   * head dim 256: one block per wave (128 key rows per workgroup), two ring stages: the only
//     kernel of that shape;
//   * head dims 64 and 128: two blocks per wave (256 key rows), four stages, beside the paired kernel
//     (dkdv_regs_is_optional below).
constexpr int dkdv_regs_blocks(int D, int dtype) {
    if (dtype == CHILL_F32) return 0;
    if (D == 256) return 1;
    return 0;
}
constexpr int dkdv_regs_stages(int D) { return D == 256 ? 2 : 4; }
// 16-bit inputs at head dims 64 and 128 have both kernels: the paired one, and dkdv_regs_kernel with two blocks per wave,
// whose runs of predicate-free tiles go through a generated loop (gen_bwd_loop.py).  The latter owns its CU (130 KiB of
// LDS, 512 registers per wave) and pays more before and after its loop (K into registers, V negated in LDS, no second
// workgroup to hide behind): it is taken for long sequences on a grid of at least two workgroups per CU, and of
// the banded masks only for those named below.  Measured on dK/dV alone, against the paired kernel:
// causal B8 H16 T8192 3.63 / 4.06 ms, B16 H16 T4096 2.18 / 2.27, B2 H8 T8192 0.547 / 0.591, full mask fp16 B4 H16
// T4096 0.98 / 1.16, prefix-LM B4 H16 T8192 1.91 / 2.16; but causal B1 H8 T8192 0.368 / 0.318, B4 H16 T2048
// 0.227 / 0.197, sliding window 512 at T8192 0.65 / 0.49.  At head dim 64 (against the 4-wave kernel that runs three
// to a CU): causal B8 H16 T4096 0.73 / 0.77, B4 H32 T8192 2.12 / 2.42, B2 H8 T8192 0.31 / 0.36, B1 H32 T16384 1.99 / 2.35,
// full mask B4 H16 T4096 0.56 / 0.73, prefix-LM B4 H32 T8192 2.12 / 2.45; there the other kernel's workgroups are a
// quarter of the size and fill a small grid better: B2 H16 T4096 (512 workgroups of this kernel) causal 0.20 / 0.17,
// prefix-LM 0.20 / 0.18 (but full mask 0.28 / 0.38); B4 H16 T4096 (1024) causal 0.37 / 0.38: from four workgroups per CU on.
constexpr int kDkdvRegsBlocks128 = 2;
// Sequence lengths from which it is taken, by what the mask leaves of a key block's loop (measured against the other
// kernel on bf16 grids of 1024 .. 4096 workgroups, B8 .. B32 H16): under a full mask every tile is predicate-free and it
// wins from the shortest sequences tried (T = 1024 / 2048 / 3072 / 4000: -16 / -17 / -18 / -17 % at head dim 128, -21 / -27 /
// -27 / -23 % at head dim 64); under a causal mask the first tiles of a key block run outside the generated loop and the
// runs shrink with the sequence (head dim 128: T = 1024 / 2048 / 3072 / 3500 / 4000 +14 / +1 / -3 / -4.5 / -5 .. -8 %;
// head dim 64: T = 2048 / 3072 / 3500 / 4000 +5 .. +17 / -2 .. +1.5 / -5 / -3 .. -5 %); prefix-LM lies between the two
// (prefix 512, head dim 128: -6 .. -10 % from T = 1024 on) and takes the causal limits; the banded masks it serves keep 4096.
constexpr int dkdv_regs_min_sequence(int mask_id, int D) {
    return mask_id == CHILL_MASK_FULL ? 1024 : mask_is_banded(mask_id) ? 4096 : D >= 128 ? 3072 : 3500;
}
constexpr int kDkdvRegsMinWorkgroups = 2 * 256;
constexpr int kDkdvRegsMinWorkgroups64 = 4 * 256;
// (by mask as well: under a full mask it wins on one workgroup per CU already, B1 H16 T4096 -24 % at head dim 128 and -38 %
// at head dim 64, where causal and prefix-LM masks lose 10-19 %; at head dim 64 the causal-like masks win on 512 workgroups
// from 8192 keys on, B1 H16 T8192 -13 %, B1 H8 T16384 -15 %, and lose 4-9 % at T = 4096)
constexpr long long dkdv_regs_min_workgroups(int mask_id, int D, int T) {
    if (mask_id == CHILL_MASK_FULL) return 256;
    if (D >= 128) return kDkdvRegsMinWorkgroups;
    return (!mask_is_banded(mask_id) && T >= 8192) ? kDkdvRegsMinWorkgroups64 / 2 : kDkdvRegsMinWorkgroups64;
}
constexpr bool dkdv_regs_is_optional(int D, int dtype) { return dtype != CHILL_F32 && (D == 128 || D == 64); }
// Banded masks take it only when a wave's 64 key rows lie in one chunk, so that its tiles are all predicate-free
// and all alike: chunkwise masks whose chunk size is a multiple of 64 (`mask_arg0` = the mask's first argument;
// measured at head dim 128, T = 8192 and 16384: chunks of 64 / 128 / 256 / 1024 rows -5 / -8 / -13 / -16 %, chunks
// of 96 rows +13 %; at head dim 64, where a tile is half the work, chunks of 64 rows +30 .. +68 %, of 128 rows +-1 %,
// of 256 rows 0 .. +8 %, of 320 rows -8 %, of 512 rows -19 %, of 1024 rows -17 %: from 320 rows on); and sliding
// windows from kDkdvRegsWideBand keys on (`band_keys` = mask_band_keys; windows of 64 .. 512 keys +32 .. +60 %,
// of 1024 +14 %, of 2048 -2 %, of 4096 -8 % at head dim 128 and -11 % at head dim 64).
constexpr int kDkdvRegsWideBand = 4096;
constexpr bool dkdv_regs_serves_band(int mask_id, long long mask_arg0, long long band_keys, int D) {
    return (mask_id == CHILL_MASK_CHUNKWISE && mask_arg0 % (32 * kDkdvRegsBlocks128) == 0 && (D >= 128 || mask_arg0 >= 320)) ||
           (mask_id == CHILL_MASK_SLIDING_WINDOW && band_keys >= kDkdvRegsWideBand);
}
// (at head dim 128 chunks of fewer than 256 rows whose band has at most 256 keys go through the workgroups that share a CU,
// dkdv_takes_one_stage, instead: bf16 B2 H16 T8192, this kernel -> that, us, 64 x 1 112 -> 84, 64 x 3 126 -> 100, 128 x 1 113 -> 92,
// 128 x 2 129 -> 118, 192 x 1 128 -> 106; B2 H32 T16384 398 -> 289, 471 -> 382, 396 -> 333, 466 -> 462, 457 -> 407.  Wider: 128 x 3
// 151 -> 140, 549 -> 575, 64 x 9 190 -> 175, 704 -> 737, 192 x 3 189 -> 177, 694 -> 752, 256 x 1 122 -> 123, 420 -> 473.  On the smallest
// grid of this kernel, 512, backward: 64 x 1 94 -> 82, 64 x 3 113 -> 104, 128 x 1 108 -> 102, 192 x 0 103 -> 93.)
constexpr bool dkdv_regs_leaves_band(int mask_id, long long mask_arg0, long long band_keys, int D) {
    return mask_id == CHILL_MASK_CHUNKWISE && D == 128 && mask_arg0 < 256 && band_keys <= 256;
}
constexpr bool dkdv_takes_regs(int mask_id, long long mask_arg0, long long band_keys, int D, long long batch_kv_heads, int T) {
    const long long workgroups = batch_kv_heads * ((T + 128 * kDkdvRegsBlocks128 - 1) / (128 * kDkdvRegsBlocks128));
    return (!mask_is_banded(mask_id) || dkdv_regs_serves_band(mask_id, mask_arg0, band_keys, D)) && T >= dkdv_regs_min_sequence(mask_id, D) &&
           workgroups >= dkdv_regs_min_workgroups(mask_id, D, T) && !dkdv_regs_leaves_band(mask_id, mask_arg0, band_keys, D);
}

// `regs`: the row of dkdv_regs_kernel where that kernel is an option (dkdv_regs_is_optional); `one_stage`: that of the paired
// kernel with a ring of one stage (dkdv_takes_one_stage)
constexpr TileConfig dkdv_tile_config(int mask_id, int D, int dtype, bool small_grid = false, bool regs = false, bool one_stage = false) {
    const int row_bytes = D * elem_bytes(dtype);
    const int blocks = (regs && dkdv_regs_is_optional(D, dtype)) ? kDkdvRegsBlocks128 : dkdv_regs_blocks(D, dtype);
    if (blocks > 0) {
        const int rows = 4 * 32 * blocks;
        return TileConfig{rows, 32, 4, rows * row_bytes + dkdv_regs_stages(D) * (2 * 32 * row_bytes + 2 * 32 * 4)};
    }
    if (dkdv_is_paired(D, dtype)) {
        const int waves = dkdv_paired_waves(mask_id, D, dtype, small_grid || one_stage);
        const int rows = 16 * waves;
        const int ring = 2 * rows * row_bytes + (one_stage ? 1 : 2) * (2 * 64 * row_bytes + 2 * 64 * 4);
        const int exchange = dkdv_paired_exchange_bytes(D) * waves / 8;
        return TileConfig{rows, 64, waves, ring > exchange ? ring : exchange};
    }
    return TileConfig{32 * dkdv_split_waves(D) / dkdv_split(D), 32, dkdv_split_waves(D), dkdv_split_lds_bytes(D, dtype)};
}

// heads = B * H, kv_heads = B * H_kv and T = sequence length of the launch (the rows of a pass depend on the heads its tiles belong
// to, in fp32 on both); T = kLongSequence for the row of long sequences on a full chip.
// mask_arg0 = the mask's first argument (the dK/dV row of chunkwise masks depends on the chunk size), band_keys =
// mask_band_keys of the mask (the forward and dK/dV rows of banded masks depend on the width of the band).
inline int tile_config(int mask_id, long long mask_arg0, long long band_keys, int D, int dtype, int pass, long long heads,
                       long long kv_heads, int T, TileConfig* out) {
    if (dtype != CHILL_F32 && dtype != CHILL_F16 && dtype != CHILL_BF16) return CHILL_ERR_BAD_DTYPE;
    if (D != 16 && D != 32 && D != 64 && D != 128 && D != 256) return CHILL_ERR_BAD_HEAD_DIM;
    if (pass != CHILL_PASS_FWD && pass != CHILL_PASS_DQ && pass != CHILL_PASS_DKDV) return CHILL_ERR_BAD_ARGUMENT;
    const long long batch_heads = pass == CHILL_PASS_DKDV ? kv_heads : heads;
    const bool small = T != kLongSequence && (pass == CHILL_PASS_FWD ? fwd_takes_small(mask_id, batch_heads, T, D, dtype)
                                                                    : bwd_takes_small(mask_id, batch_heads, T, D, dtype, pass));
    const bool parts = f32_takes_parts(band_keys, heads, kv_heads, T, D, dtype);
    if (small && !(parts && f32_takes_group(batch_heads, T, D))) {
        const int lds = pass == CHILL_PASS_FWD ? fwd_small_lds_bytes(D, dtype) : bwd_small_lds_bytes(D, dtype, pass == CHILL_PASS_DQ ? 1 : 2, parts);
        *out = small_tile_config(mask_id, dtype, pass, lds, batch_heads * ((T + 31) / 32), T, band_keys);
        return CHILL_OK;
    }
    if (parts) {
        *out = f32_group_tile_config(D, pass);
        return CHILL_OK;
    }
    switch (pass) {
        case CHILL_PASS_FWD:
            *out = fwd_tile_config(mask_id, D, dtype, fwd_takes_short_row(mask_id, band_keys, batch_heads, T) ? 1 : kLongSequence);
            return CHILL_OK;
        case CHILL_PASS_DQ:
            if (dq_regs2_is_optional(D, dtype) && (T == kLongSequence ? !mask_is_banded(mask_id) : dq_takes_regs2(mask_id, batch_heads, T))) {
                *out = dq_regs2_tile_config(D, dtype);
                return CHILL_OK;
            }
            *out = dq_tile_config(mask_id, D, dtype, (T != kLongSequence && dq_takes_short_row(batch_heads, T)) ? 1 : kLongSequence);
            return CHILL_OK;
        case CHILL_PASS_DKDV: {
            // (the row of long sequences on a full chip: the generated loop where there is one)
            const bool is_long = T == kLongSequence;
            const bool regs = dkdv_regs_is_optional(D, dtype) &&
                              (is_long ? (!mask_is_banded(mask_id) || dkdv_regs_serves_band(mask_id, mask_arg0, band_keys, D))
                                       : dkdv_takes_regs(mask_id, mask_arg0, band_keys, D, batch_heads, T));
            const bool small_row = !regs && !is_long && dkdv_takes_small_row(mask_id, batch_heads, T);
            const bool one_stage = !regs && !small_row && dkdv_one_stage_serves(mask_id, D, dtype) &&
                                   dkdv_takes_one_stage(mask_id, band_keys, batch_heads, is_long ? 1 : T, false);
            *out = dkdv_tile_config(mask_id, D, dtype, small_row, regs, one_stage);
            return CHILL_OK;
        }
        default: return CHILL_ERR_BAD_ARGUMENT;
    }
}

// Work-item order: workgroups are dealt round-robin to the 8 XCDs (each with its own L2), so the
// linear workgroup id is remapped to give every XCD a contiguous run of work items.  Returns the
// work item index or -1 when this workgroup has nothing to do.
//
// `resident` = workgroups of the kernel that share a CU.  A grid that the chip holds at once (more workgroups than CUs,
// at most `resident` per CU) is placed statically: the dispatcher deals an XCD's workgroups to its 32 CUs pass after
// pass in the same CU order, so workgroup l of an XCD and workgroup l + 32 share a CU.  The kernels order their
// work items longest first (under causal-like masks a tile's work grows with its index), which would hand a CU the
// longest items of both passes and another the shortest; every second pass is therefore taken in reverse, and the two
// items of a CU add up alike (measured on dq_kernel, 512 workgroups of four waves, causal bf16 at head dim 128:
// B1 H16 T4096 148 -> 113 us, B1 H32 T2048 82 -> 66, B2 H8 T4096 147 -> 116, B1 H8 T8192 216 -> 204).  Larger grids
// are dealt out as CUs become free, and longest first is the right order for that.
CHILL_HD int xcd_contiguous_item(int wg, int total, int resident = 1) {
    constexpr int kXcds = 8, kCusPerXcd = 32;
    const int per = (total + kXcds - 1) / kXcds;
    const int first = (wg % kXcds) * per;
    int local = wg / kXcds;
    if (resident > 1 && total > kXcds * kCusPerXcd && total <= resident * kXcds * kCusPerXcd) {
        const int pass = local / kCusPerXcd;
        if (pass & 1) {
            const int valid = total - first < per ? total - first : per;  // items of this XCD
            const int len = valid - pass * kCusPerXcd < kCusPerXcd ? valid - pass * kCusPerXcd : kCusPerXcd;
            const int c = local - pass * kCusPerXcd;
            if (c < len) local = pass * kCusPerXcd + len - 1 - c;
        }
    }
    const int item = first + local;
    return (local < per && item < total) ? item : -1;
}

// The order in which a launch's workgroups take their (head, tile) items, as the number of heads of a BLOCK: the blocks
// follow each other, inside one the workgroups take tile 0 of every head, then tile 1 of every head, and so on, and the
// heads keep to their XCDs as work_item says.  The kernels number a head's tiles from the heavy end of a causal-like
// mask, so a block, the last one above all, ends with its short tiles; a whole launch as one block is longest first, but
// streams the K and V (in dK/dV the Q and dO) of all its heads at once through an XCD's L2 (4 MiB) and the last-level
// cache (256 MiB).  So a block holds as many heads per XCD as stream about 16 MiB, two at the least.
// 0: every XCD takes a contiguous run of heads, one after the other (xcd_contiguous_item).
// Measured, forward / dQ / dK/dV in us, contiguous runs -> blocks of this size (bf16):
//   causal D128 B4 H32/8 T2085    205 / 233 / 354 -> 172 / 214 / 288      causal D64 B4 H16 T4096  144 / 222 / 327 -> 143 / 191 / 284
//   causal D128 B8 H16 T4096  488 / 755 / 1060 -> 488 / 717 / 988         causal D128 B8 H16 T8192 1741 / 2560 / 3435 -> 1735 / 2506 / 3350
//   (D128 B8 H16 as one block: T4096 501 / 747 / 998, T8192 1878 / 2660 / 3518)
//   causal D256 B4 H8 T2048 87 / 158 / 227 -> 86 / 113 / 155; full mask fp16 D64 B8 H12 T4042 469 / 579 / 724 -> 433 / 576 / 725
// The forward, whose pairs of q-tiles are all of the same length, has nothing to balance and takes half of that (causal
// D128 B8 H16 T8192: 1735 with two heads per XCD, 1748 with four).  Banded masks, whose tiles are all alike and share
// their keys with the next tile, keep the contiguous runs (within 2 % either way).
// A padded batch: the work of a head depends on its batch element, and contiguous runs gave the long elements to some
// XCDs and the short ones to others.  Two heads per XCD, the elements longest first (batch_by_length): the order that
// was never far from the best over blocks of 1, 2, 4, 8 and all heads, lengths of T/4 .. T, unsorted or sorted: causal
// D128 B4 H32/8 T2085 197 / 219 / 340 -> 116 / 139 / 210, B8 H16 T8192 1456 / 2199 / 2935 -> 969 / 1368 / 1830,
// full mask B8 H16 T2085 303 / 348 / 446 -> 172 / 229 / 290, sliding window 128 + 128 B8 H16 T4042 154 / 183 / 271 ->
// 127 / 158 / 217.
// `es` = bytes of an element; the heads of a launch are query heads, in dK/dV key / value heads, and `streams` of them
// share what they stream (work_streams).
constexpr long long kWorkBlockBytes = 16ll << 20;
constexpr int work_streams(int pass, int H, int H_kv) { return pass == CHILL_PASS_DKDV ? 1 : H / H_kv; }
constexpr int work_block(int mask_id, int pass, bool padded, int B, int H, int H_kv, int T, int D, int es) {
    if (!padded && mask_is_banded(mask_id)) return 0;
    const int streams = work_streams(pass, H, H_kv);
    const long long sets = (long long)B * H_kv, rounds = (sets + 7) / 8;  // sets per XCD
    const long long bytes = 2ll * T * D * es * (pass == CHILL_PASS_DKDV ? H / H_kv : 1);
    const long long budget = (pass == CHILL_PASS_FWD ? kWorkBlockBytes / 2 : kWorkBlockBytes) / bytes;
    const long long most = padded || budget < 2 ? 2 : budget;
    const long long blocks = rounds / most < 1 ? 1 : rounds / most;
    return (int)((rounds + blocks - 1) / blocks * 8 * streams);
}

// The same for the device: as many blocks as that makes, equal up to one round, because a last block of fewer heads would
// end the launch on a part of the CUs.  The smaller blocks come first, and an incomplete round goes with the first of them.
// (causal D128: B4 H32/8 T2085, dK/dV, one block of four heads per XCD 290 us, three and one 373.  Forward / dQ / dK/dV,
// the last block what is left over -> equal blocks: B2 H25 T6000 453 / 587 / 808 -> 386 / 586 / 803, B8 H16 T6000 1000 /
// 1453 / 1942 -> 1000 / 1463 / 1966, B8 H32 T6000 1995 / 2945 / 3927 -> 1992 / 2922 / 3916; padded, lengths of T/4 .. T,
// B13 H8 T4096 240 / 322 / 463 -> 238 / 320 / 454, B5 H9 T4096 141 / 179 / 277 -> 133 / 173 / 254.)
// A padded launch takes the heads of a block of no whole number of rounds in turn: with sets that keep to their XCDs some
// XCDs get the long elements and others the short ones (causal D128 B3 H32/4, lengths 4096, 3000 and 1024, forward / dQ /
// dK/dV: 214 / 288 / 720 us in turn, 264 / 366 / 756 in groups).
constexpr WorkOrder work_order(bool padded, long long heads, int streams, int block) {
    if (block == 0) return WorkOrder{0, 0, 0};
    const long long sets = heads / streams, rounds = sets / 8;
    const long long most = block < 16ll * streams ? 1 : block / (8ll * streams);  // rounds of a block
    const long long wanted = ((sets + 7) / 8 + most - 1) / most;
    const long long blocks = wanted > rounds ? (rounds > 1 ? rounds : 1) : wanted;
    return WorkOrder{(int32_t)(blocks - rounds % blocks), (int32_t)(rounds / blocks * 8), (int32_t)(sets % 8) + (padded ? 8 : 0)};
}

// Workgroup `wg` of a launch of `heads` heads (query heads, or key / value heads in dK/dV; `streams` of them share what
// they stream, a set) of `per_head` tiles each, in the order `order`: its head and tile, or false if it has nothing to do.
// `resident` as in xcd_contiguous_item.
// Workgroups are dealt round-robin to the XCDs.  The sets of a block are taken in groups of 1, 2 and 4, the bits of their
// number modulo 8, and one of the rest, a multiple of 8; inside a group of n the workgroups alike modulo min(n, 8), the
// same ones for every tile, take the same sets.  So a set of the large group stays on one XCD, one of a small group on
// 8 / n of them, and an XCD streams one set of each small group, whatever the number of heads (with the heads of a tile
// simply in turn it streams all 25 of B1 H25).  Measured, forward / dQ / dK/dV in us, in turn -> in groups (bf16):
//   causal D64  B1 H25 T8192 227 / 296 / 405 -> 214 / 292 / 403   B1 H12 T4042 41 / 59 / 71 -> 39 / 58 / 72
//               B1 H5 T4042  40.3 / 56.0 / 59.0 -> 35.8 / 55.2 / 59.0   full D64 B5 H5 T1500 27.6 / 35.8 / 48.1 -> 27.0 / 35.1 / 45.8
//   causal D128 B1 H15 T8192 216 / 324 / 466 -> 215 / 325 / 466   B3 H28/4 T4096 331 / 462 / 745 -> 328 / 464 / 743
// Contiguous runs keep the sets together as well and are slower than both where tiles differ (B1 H25: 241 / 351 / 456; H15:
// 296 / 477 / 549; under a full mask, fp16 B1 H25, 451 / 633 / 864 against 451 / 627 / 862).  The small groups ahead of the
// blocks instead of inside them, tile by tile, lose what longest first gains (H15: 244 / 375 / 514).
CHILL_HD bool work_item(int wg, int heads, int per_head, WorkOrder order, int streams, int resident, int* head, int* tile) {
    constexpr int kXcds = 8, kCusPerXcd = 32;
    const int total = heads * per_head;
    if (order.small == 0) {
        const int item = xcd_contiguous_item(wg, total, resident);
        if (item < 0) return false;
        *head = item / per_head;
        *tile = item - *head * per_head;
        return true;
    }
    if (wg >= total) return false;
    if (resident > 1 && total > kXcds * kCusPerXcd && total <= resident * kXcds * kCusPerXcd) {
        const int xcd = wg % kXcds, local = wg / kXcds, pass = local / kCusPerXcd;
        const int mine = (total - xcd + kXcds - 1) / kXcds;  // items of this XCD
        if (pass & 1) {
            const int len = mine - pass * kCusPerXcd < kCusPerXcd ? mine - pass * kCusPerXcd : kCusPerXcd;
            wg = (pass * kCusPerXcd + len - 1 - (local - pass * kCusPerXcd)) * kXcds + xcd;
        }
    }
    // (all of it is non-negative: unsigned divisions are the shorter ones)
    const unsigned w = wg, rest = order.rest % kXcds, set_items = streams * per_head;
    unsigned first = 0, sets = order.sets + rest;  // first set and number of sets of the block
    if (w >= sets * set_items) {
        unsigned later = w - sets * set_items;  // items since the end of the first block
        first = sets;
        sets = order.sets;
        const unsigned small_items = (order.small - 1) * sets * set_items;
        if (later >= small_items) {
            later -= small_items;
            first += (order.small - 1) * sets;
            sets += 8;
        }
        first += later / (sets * set_items) * sets;
    }
    const unsigned size = sets * streams, i = w - first * set_items;
    *tile = i / size;
    unsigned in_group = i - *tile * size;
    unsigned before = 0, shift = 3;  // sets of the block's groups before this one; min(n, 8) = 1 << shift
    if (rest > 0 && first == 0) {
        if (order.rest >= kXcds) {
            *head = in_group;
            return true;
        }
        if (in_group < rest * streams)
            for (shift = 0; !(rest >> shift & 1) || in_group >= (before + (1 << shift)) * streams; shift++) before += rest & 1 << shift;
        else
            before = rest;
        in_group -= before * streams;
    }
    const unsigned k = in_group >> shift, round = streams > 1 ? k / streams : k;  // (the heads of a set follow each other)
    const unsigned set = first + before + (w & ((1 << shift) - 1)) + (round << shift);
    *head = set * streams + k - round * streams;
    return true;
}

}  // namespace chill
