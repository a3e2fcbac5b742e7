// Forward, dQ and dK/dV of fp32 inputs on the fp16 matrix instructions (chill_f32_parts.h), rows of at most 512 bytes.
//
// A workgroup owns R row tiles of 32 rows (queries in the forward and dQ, keys in dK/dV) of one head, its members, and walks the
// 32-row blocks of the other axis in S streams: stream s takes the blocks s, s + S, ...  Every (member, stream) is a wave with
// accumulators of its own; the S partial results of a member are merged through LDS at the end (the forward's like the parts of
// a softmax, the gradients are sums).  The R waves of a stream share its blocks: each brings its share of a block from global
// memory through registers to LDS, scaled and split, while the block before is worked on, one workgroup barrier per block.
// R = 4 serves full grids, R = 2 launches of few tiles (under masks whose rows grow with their index its two members are the
// j-th tile from either end, so that all workgroups have the same work, and share the blocks both see), R = 1 launches of fewer
// tiles than CUs; f32_shape (chill_tiles.h) has the lines and what was measured.
// What bounds it: at head dim 64 a block of the forward costs a SIMD about 2200 cycles of which 768 are its 24 MFMAs; the
// others are vector instructions (about 100 for a share of the next block, 90 for the softmax, 50 for P), which hardly overlap with
// MFMAs.  Full grids run at 270 TFLOP/s of fp32 products in the forward and 250 in dK/dV, where the fp32 instruction, whose
// peak is 157, reached 118 and 105 (causal B4 H16 T4096: forward 1160 -> 509 us, dQ 1680 -> 659, dK/dV 2210 -> 925).
//
// Every sum is finite unless an input is not (or the true result overflows): a wave that ends with a sum that is not computes
// its blocks again with the fp32 matrix instruction, straight from global memory (native_*), which is what defines the result.
#pragma once

#include "chill_device.h"
#include "chill_f32_parts.h"
#include "chill_mask.h"
#include "chill_params.h"
#include "chill_tiles.h"

namespace chill {

// ---------------------------------------------------------------- the fp32 instruction, operands from global memory
// X (32 rows) B^T (32 rows), both row-wise
template <int D>
__device__ __forceinline__ f32x16 native_rowwise(const float* x, int64_t x_stride, int x_rows, const float* b, int64_t b_stride,
                                                 int b_rows, int lane) {
    const int n = lane & 31, h = lane >> 5;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll 2
    for (int j = 0; j < D / 8; j++) {
        i32x4 xv = {0, 0, 0, 0}, bv = {0, 0, 0, 0};
        if (n < x_rows) xv = *reinterpret_cast<const i32x4*>(x + (int64_t)n * x_stride + 4 * (2 * j + h));
        if (n < b_rows) bv = *reinterpret_cast<const i32x4*>(b + (int64_t)n * b_stride + 4 * (2 * j + h));
        acc = Elem<f32_t>::mma(xv, bv, acc);
    }
    return acc;
}
// acc += X^T P, X 32 rows, P an accumulator block; the head-dim blocks from `db0` on
template <int D, int N>
__device__ __forceinline__ void native_transposed(const float* x, int64_t x_stride, int x_rows, const f32x16& p, f32x16 (&acc)[N],
                                                  int lane, int db0 = 0) {
    const int n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = 8 * (r / 4) + 4 * h + (r % 4);
#pragma unroll
        for (int db = 0; db < N; db++) {
            const int col = D < 32 ? (n & (D - 1)) : 32 * (db0 + db) + n;
            const float a = row < x_rows ? x[(int64_t)row * x_stride + col] : 0.f;
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, p[r], acc[db], 0, 0, 0);
        }
    }
}

// ---------------------------------------------------------------- work of a workgroup
// Member `m` of group `j` (0: the heavy end) of a head's n tiles, or -1.
template <int MASK, int R, int S, bool QROWS>
struct F32Group {
    static constexpr bool kMirrored = R == 2 && S > 1 && mask_rows_grow(MASK);
    int tile0, j, n;
    __device__ __forceinline__ F32Group(int group, int n_tiles) : j(group), n(n_tiles) {
        tile0 = R * (QROWS ? (n_tiles + R - 1) / R - 1 - group : group);
    }
    __device__ __forceinline__ int tile(int m) const {
        if (kMirrored) {
            const int far = n - 1 - j, t = (m == 0) == QROWS ? far : j;
            return (m == 0 || far != j) ? t : -1;
        }
        return tile0 + m < n ? tile0 + m : -1;
    }
    // the blocks any member visits
    __device__ __forceinline__ Range hull(int seq_len, MaskArgs a) const {
        if (kMirrored) {
            Range out = {0x7fffffff, 0};
            for (int m = 0; m < 2; m++) {
                const int t = tile(m);
                if (t < 0 || 32 * t >= seq_len) continue;
                const TileRange r = tile_range<MASK, QROWS>(32 * t, 32, 32, seq_len, false, a);
                if (r.start < r.end) out = Range{imin(out.lo, r.start), imax(out.hi, r.end)};
            }
            return out;
        }
        if (32 * tile0 >= seq_len) return {0, 0};
        const TileRange r = tile_range<MASK, QROWS>(32 * tile0, 32 * R, 32, seq_len, false, a);
        return {r.start, r.end};
    }
};

// LDS of a workgroup: [stage][stream] two PartTiles (one stage where a wave has its blocks to itself) and, behind them,
// [stage][stream] the fields of their scales (and in dK/dV LSE2 and delta of the block's rows).
template <int D, int R, int S, int PASS>
struct F32Lds {
    static constexpr int VEC = PASS == CHILL_PASS_DKDV ? 64 : 0;
    static constexpr int TILE = PartTile<D>::BYTES;
    static constexpr int SLICES = R >= 2 ? R / 2 : 1;  // of a tile, one per wave
    static constexpr int TENSORS = R >= 2 ? 1 : 2;     // tiles a wave has a share of
    static constexpr int STAGES = R >= 2 ? 2 : 1;
    static constexpr int FIELDS = STAGES * S * 2 * TILE;
    static constexpr int VECS = FIELDS + STAGES * S * 2 * SLICES * 4;
    static constexpr int BYTES = f32_lds_bytes(D, R, S, PASS);
    static_assert(VECS + STAGES * S * VEC * 4 <= BYTES, "the ring fits");
    char* base;
    int stream;
    __device__ __forceinline__ char* tile(int stage, int tensor) const { return base + ((stage * S + stream) * 2 + tensor) * TILE; }
    __device__ __forceinline__ int* fields(int stage, int tensor) const {
        return reinterpret_cast<int*>(base + FIELDS) + ((stage * S + stream) * 2 + tensor) * SLICES;
    }
    __device__ __forceinline__ float* vec(int stage) const { return reinterpret_cast<float*>(base + VECS) + (stage * S + stream) * VEC; }
    __device__ __forceinline__ void read_fields(int stage, int tensor, int (&out)[SLICES]) const {
#pragma unroll
        for (int i = 0; i < SLICES; i++) out[i] = uniform(fields(stage, tensor)[i]);
    }
};

// waves per SIMD a kernel is compiled for: two where two workgroups of four waves, or one of eight, share a CU
constexpr int f32_waves_per_simd(int members, int waves, int lds_bytes) {
    return (waves >= 8 || (members > 1 && 2 * lds_bytes <= 160 * 1024)) ? 2 : 1;
}

// x[r] *= the inverse of its row's scale, times f
template <int SLICES>
__device__ __forceinline__ void unscale_factors(const int (&field)[SLICES], float f, float (&out)[SLICES]) {
#pragma unroll
    for (int i = 0; i < SLICES; i++) out[i] = parts_inverse(field[i]) * f;
}

// The mask of a block that is not predicate-free: entries no pair sees become `fill`.  `pos` = the lane's own row or key.
template <int MASK, bool QROWS>
__device__ __forceinline__ void mask_f32_block(f32x16& s, const Range& vis, int pos, int other0, int seq_len, MaskArgs a, int h,
                                               float fill) {
    if constexpr (Mask<MASK>::kRowIsRange) {
        fill_outside_range(s, vis.lo, vis.hi, other0 + 4 * h, fill);
    } else {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int other = other0 + 8 * (r / 4) + 4 * h + (r % 4);
            const int q = QROWS ? pos : other, k = QROWS ? other : pos;
            s[r] = (q < seq_len && k < seq_len && Mask<MASK>::pred(q, k, seq_len, a)) ? s[r] : fill;
        }
    }
}

// ---------------------------------------------------------------- forward
template <int D, int MASK, int R, int S>
__global__ __launch_bounds__(R * S * 64)
__attribute__((amdgpu_waves_per_eu(f32_waves_per_simd(R, R * S, F32Lds<D, R, S, CHILL_PASS_FWD>::BYTES))))
void fwd_f32_kernel(FwdParams p, int n_tiles, int n_groups, int has_full_blocks) {
    typedef F32Lds<D, R, S, CHILL_PASS_FWD> Lds;
    constexpr int DB = (D + 31) / 32, NSL = Lds::SLICES;
    constexpr int kAhead = D >= 128 ? 2 : 4;  // operands of the last products read ahead
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, j;
    if (!work_item(blockIdx.x, p.B * p.H, n_groups, order_of(p), p.group, 1, &bh, &j)) return;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H);
    const int hd = bh % p.H, hkv = hd / p.group;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int stream = wave % S, member = wave / S;
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const F32Group<MASK, R, S, true> group(j, n_tiles);
    const Range hull = group.hull(seq_len, p.margs);
    const int n_iters = hull.hi > hull.lo ? (hull.hi - hull.lo + S - 1) / S : 0;
    const int tile = group.tile(member);
    const int qb = 32 * (tile < 0 ? 0 : tile);
    const int q_pos = qb + n;
    TileRange wr = {0, 0, 0, 0};
    if (tile >= 0 && qb < seq_len) wr = tile_range_rows_discarded<MASK, true>(qb, 32, 32, seq_len, has_full_blocks != 0, p.margs);

    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h + (int64_t)qb * p.sq.t;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    // this wave's share of its stream's blocks
    const Lds lds = {smem, stream};
    const int slice = member % NSL, my_tensor = R >= 2 ? member / NSL : 0;
    PartStager<D, 32 / NSL> rows[Lds::TENSORS];
    bool fetched = false;
    auto fetch = [&](int it) {
        const int row0 = 32 * (hull.lo + it * S + stream) + slice * (32 / NSL);
        fetched = it < n_iters && row0 < 32 * hull.hi;
        if (!fetched) return;
#pragma unroll
        for (int i = 0; i < Lds::TENSORS; i++) {
            const bool is_v = my_tensor + i == 1;
            rows[i].fetch(is_v ? vptr : kptr, is_v ? p.sv.t : p.sk.t, row0, seq_len, lane);
        }
    };
    // what was fetched to LDS, as block `it`: first its scale, then the parts, in STEPS shares
    constexpr int STEPS = PartStager<D, 32 / NSL>::STEPS * Lds::TENSORS;
    auto measure = [&](int it) {
        if (!fetched) return;
#pragma unroll
        for (int i = 0; i < Lds::TENSORS; i++) {
            rows[i].measure();
            if (lane == 0) lds.fields(it % Lds::STAGES, my_tensor + i)[slice] = rows[i].field;
        }
    };
    auto commit = [&](int it, auto step) {
        constexpr int i = decltype(step)::value % Lds::TENSORS, share = decltype(step)::value / Lds::TENSORS;
        if constexpr (decltype(step)::value < STEPS)
            rows[i].template commit<share>(lds.tile(it % Lds::STAGES, my_tensor + i), slice * (32 / NSL), lane);
    };
    auto commit_all = [&](int it) {
        if (!fetched) return;
        measure(it);
        static_for<STEPS>([&](auto step) { commit(it, step); });
    };
    fetch(0);
    ResidentParts<D> qf;
    // a negative scale reverses the order of the scores: its sign goes into Q
    qf.load(qptr, p.sq.t, tile >= 0 ? seq_len - qb : 0, lane, p.scale_log2 < 0.f ? -1.f : 1.f);
    OperandOffsets<f16_t, D> ofs;
    ofs.init(lane);
    commit_all(0);
    fetch(1);

    f32x16 o[DB];
    float m_run = -INFINITY;  // running max of the row over this wave's keys (scaled, log2 domain)
    float l_run = 0.f;        // this lane's share of the row sum
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < DB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[i][r] = 0.f;
        m_run = -INFINITY;
        l_run = 0.f;
    };
    clear();
    const Range vis = visible_range<MASK, true>(q_pos, seq_len, p.margs);
    const float scale = fabsf(p.scale_log2);
    // one block's online softmax (chill_fwd.py:214-226) of s times f, f per slice of its rows; a row that has seen no key keeps 0
    // as its reference
    auto softmax = [&](f32x16& s, auto& f, int blk) {
        constexpr int N = sizeof(f) / sizeof(f[0]);
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, true>(s, vis, q_pos, blk * 32, seq_len, p.margs, h, -INFINITY);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < N; i++) {
            float part = s[16 / N * i];
#pragma unroll
            for (int r = 1; r < 16 / N; r++) part = fmaxf(part, s[16 / N * i + r]);
            mx = fmaxf(mx, part * f[i]);
        }
        mx = max_across_halves(mx);
        const float m_new = fmaxf(m_run, mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
            const float alpha = fast_exp2(((m_run == -INFINITY) ? 0.f : m_run) - m_use);
            l_run *= alpha;
            scale_blocks(o, alpha);
            m_run = m_new;
        }
        float psum[2] = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = fast_exp2(__builtin_fmaf(s[r], f[r * N / 16], -m_use));
            psum[r % 2] += s[r];
        }
        l_run += psum[0] + psum[1];
    };

    ProbabilitySum sum;
    for (int it = 0; it < n_iters; it++) {
        if constexpr (R > 1) __syncthreads();  // block `it` is in LDS; everyone is done with the block before
        const int stage = it % Lds::STAGES, blk = hull.lo + it * S + stream;
        const bool mine = blk >= wr.start && blk < wr.end;
        if (mine) {
            // beside the score MFMAs the next block's scale is found, beside those of O^T it is split (one past the end: rows
            // that nobody reads)
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            s = mma_rowwise_parts<D>((const lds_char*)lds.tile(stage, 0), ofs, qf, s, lane, [&](auto t) {
                if constexpr (R > 1 && t == 0) measure(it + 1);
            });
            TransposedParts<D, kAhead> vt((const lds_char*)lds.tile(stage, 1), ofs, lane);
            vt.begin();
            int k_field[NSL], v_field[NSL];
            lds.read_fields(stage, 0, k_field);
            lds.read_fields(stage, 1, v_field);
            float f[NSL];
            unscale_factors(k_field, qf.inverse * scale, f);
            // (a factor that underflows belongs to scores of zero; as zero it would make NaN of the masked ones' -inf)
#pragma unroll
            for (int i = 0; i < NSL; i++) f[i] = fmaxf(f[i], 0x1p-126f);
            softmax(s, f, blk);
            sum.scales(v_field, o, f);
            vt.run(s, f, o, [&](auto u) {  // O^T += V^T P^T
                constexpr int PER = (STEPS + 2 * DB - 1) / (2 * DB);
                if constexpr (R > 1) static_for<PER>([&](auto e) { commit(it + 1, std::integral_constant<int, u * PER + e>{}); });
            });
        } else if (R > 1) {
            commit_all(it + 1);
        }
        if (R > 1) fetch(it + 2);
        if (R == 1) {
            commit_all(it + 1);
            fetch(it + 2);
        }
    }
    sum.finish(o);
    if (__builtin_amdgcn_ballot_w64(finite_probe(o, l_run * 0.f) != 0.f) != 0) {
        clear();
        for (int blk = hull.lo + stream; blk < wr.end; blk += S) {
            if (blk < wr.start) continue;
            const int k0 = blk * 32;
            f32x16 s = native_rowwise<D>(kptr + k0 * p.sk.t, p.sk.t, seq_len - k0, qptr, p.sq.t, seq_len - qb, lane);
            float f[1] = {scale};
            if (p.scale_log2 < 0.f) {
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] = -s[r];
            }
            softmax(s, f, blk);
            native_transposed<D>(vptr + k0 * p.sv.t, p.sv.t, seq_len - k0, s, o, lane);
        }
    }

    // ---- merge the streams' partial results
    float l_row = sum_across_halves(l_run);
    if constexpr (S > 1) {
        constexpr int PART = DB * 16 * 64;  // floats of a wave's O^T; then m and l of its lanes
        float* mine = reinterpret_cast<float*>(smem) + wave * (PART + 128);
        static_assert(R * S * (PART + 128) * 4 <= Lds::BYTES, "the partial results fit");
        __syncthreads();  // everyone is done with the tiles
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int r = 0; r < 16; r++) mine[(db * 16 + r) * 64 + lane] = o[db][r];
        mine[PART + lane] = m_run;
        mine[PART + 64 + lane] = l_row;
        __syncthreads();
        if (tile < 0 || q_pos >= p.T) return;
        const float* first = reinterpret_cast<const float*>(smem) + member * S * (PART + 128);
        float m_all = -INFINITY;
#pragma unroll
        for (int w = 0; w < S; w++) m_all = fmaxf(m_all, first[w * (PART + 128) + PART + lane]);
        const float m_ref = (m_all == -INFINITY) ? 0.f : m_all;
        float weight[S], l_all = 0.f;
#pragma unroll
        for (int w = 0; w < S; w++) {
            const float* ml = first + w * (PART + 128) + PART;
            weight[w] = (ml[lane] == -INFINITY) ? 0.f : fast_exp2(ml[lane] - m_ref);
            l_all += ml[64 + lane] * weight[w];
        }
        const bool valid = q_pos < seq_len;
        const float l_safe = (l_all == 0.f) ? 1.f : l_all;
        const float inv = 1.f / l_safe;
        float* orow = reinterpret_cast<float*>(p.o) + b * p.so.b + hd * p.so.h + (int64_t)q_pos * p.so.t;
        // wave `stream` of a member finishes every S-th group of four columns d0 .. d0 + 3 of the lane's row
        for (int u = stream; u < 4 * DB; u += S) {
            const int d0 = 8 * u + 4 * h;
            if (D < 32 && d0 >= D) continue;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < S; w++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[e] += first[w * (PART + 128) + (4 * u + e) * 64 + lane] * weight[w];
#pragma unroll
            for (int e = 0; e < 4; e++) acc[e] = valid ? acc[e] * inv : 0.f;
            *reinterpret_cast<f32x4*>(orow + d0) = acc;
        }
        // LSE2 = m + log2(l) (chill_fwd.py:288-289); -inf for a row that saw no key, 0 for rows past lens
        if (p.lse != nullptr && stream == 0 && h == 0)
            p.lse[b * p.lse_b + hd * p.lse_h + q_pos] = valid ? m_all + __log2f(l_safe) : 0.f;
    } else {
        if (tile < 0 || q_pos >= p.T) return;
        const bool valid = q_pos < seq_len;
        const float l_safe = (l_row == 0.f) ? 1.f : l_row;
        float* orow = reinterpret_cast<float*>(p.o) + b * p.so.b + hd * p.so.h + (int64_t)q_pos * p.so.t;
        store_row_transposed<f32_t, D>(orow, o, 1.f / l_safe, valid, h);
        if (p.lse != nullptr && h == 0) p.lse[b * p.lse_b + hd * p.lse_h + q_pos] = valid ? m_run + __log2f(l_safe) : 0.f;
    }
}

// ---------------------------------------------------------------- the partial gradients of a member's streams
// `acc` = OUT accumulators of DB blocks; sums over the member's S waves, scaled, to rows of `out`.
template <int D, int R, int S, int OUT, int LDS_BYTES>
__device__ __forceinline__ void f32_store_gradients(char* smem, const f32x16* const (&acc)[OUT], float* const (&row)[OUT],
                                                    const float (&mult)[OUT], int wave, int lane, bool in_tensor, bool valid) {
    constexpr int DB = (D + 31) / 32, PART = DB * 16 * 64;
    const int member = wave / S, stream = wave % S, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < OUT; i++) {
        if constexpr (S > 1) {
            static_assert(R * S * PART * 4 <= LDS_BYTES, "the partial results fit");
            __syncthreads();  // everyone is done with the tiles, or with the accumulators before
            float* mine = reinterpret_cast<float*>(smem) + wave * PART;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) mine[(db * 16 + r) * 64 + lane] = acc[i][db][r];
            __syncthreads();
            if (!in_tensor) continue;
            const float* first = reinterpret_cast<const float*>(smem) + member * S * PART;
            for (int u = stream; u < 4 * DB; u += S) {
                const int d0 = 8 * u + 4 * h;
                if (D < 32 && d0 >= D) continue;
                f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < S; w++)
#pragma unroll
                    for (int e = 0; e < 4; e++) x[e] += first[w * PART + (4 * u + e) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = valid ? x[e] * mult[i] : 0.f;
                *reinterpret_cast<f32x4*>(row[i] + d0) = x;
            }
        } else if (in_tensor) {
#pragma unroll
            for (int u = 0; u < 4 * DB; u++) {
                const int d0 = 8 * u + 4 * h;
                if (D < 32 && d0 >= D) continue;
                f32x4 x;
#pragma unroll
                for (int e = 0; e < 4; e++) x[e] = valid ? acc[i][u / 4][4 * (u % 4) + e] * mult[i] : 0.f;
                *reinterpret_cast<f32x4*>(row[i] + d0) = x;
            }
        }
    }
}

// ---------------------------------------------------------------- dQ
template <int D, int MASK, int R, int S>
__global__ __launch_bounds__(R * S * 64)
__attribute__((amdgpu_waves_per_eu(D >= 128 ? 1 : f32_waves_per_simd(R, R * S, F32Lds<D, R, S, CHILL_PASS_DQ>::BYTES))))
void dq_f32_kernel(BwdParams p, int n_tiles, int n_groups, int has_full_blocks) {
    typedef F32Lds<D, R, S, CHILL_PASS_DQ> Lds;
    constexpr int DB = (D + 31) / 32, NSL = Lds::SLICES;
    constexpr int kAhead = D >= 128 ? 2 : 4;  // operands of the last products read ahead
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, j;
    if (!work_item(blockIdx.x, p.B * p.H, n_groups, order_of(p), p.group, 1, &bh, &j)) return;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H);
    const int hd = bh % p.H, hkv = hd / p.group;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int stream = wave % S, member = wave / S;
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const F32Group<MASK, R, S, true> group(j, n_tiles);
    const Range hull = group.hull(seq_len, p.margs);
    const int n_iters = hull.hi > hull.lo ? (hull.hi - hull.lo + S - 1) / S : 0;
    const int tile = group.tile(member);
    const int qb = 32 * (tile < 0 ? 0 : tile);
    const int q_pos = qb + n;
    const int q_rows = tile >= 0 ? p.T - qb : 0, q_seen = tile >= 0 ? seq_len - qb : 0;  // (of the tensor, of the sequence)
    TileRange wr = {0, 0, 0, 0};
    if (tile >= 0 && qb < seq_len) wr = tile_range_rows_discarded<MASK, true>(qb, 32, 32, seq_len, has_full_blocks != 0, p.margs);

    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h + (int64_t)qb * p.sq.t;
    const float* doptr = reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hd * p.sdo.h + (int64_t)qb * p.sdo.t;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    const Lds lds = {smem, stream};
    const int slice = member % NSL, my_tensor = R >= 2 ? member / NSL : 0;
    PartStager<D, 32 / NSL> rows[Lds::TENSORS];
    bool fetched = false;
    auto fetch = [&](int it) {
        const int row0 = 32 * (hull.lo + it * S + stream) + slice * (32 / NSL);
        fetched = it < n_iters && row0 < 32 * hull.hi;
        if (!fetched) return;
#pragma unroll
        for (int i = 0; i < Lds::TENSORS; i++) {
            const bool is_v = my_tensor + i == 1;
            rows[i].fetch(is_v ? vptr : kptr, is_v ? p.sv.t : p.sk.t, row0, seq_len, lane);
        }
    };
    // what was fetched to LDS, as block `it`: first its scale, then the parts, in STEPS shares
    constexpr int STEPS = PartStager<D, 32 / NSL>::STEPS * Lds::TENSORS;
    auto measure = [&](int it) {
        if (!fetched) return;
#pragma unroll
        for (int i = 0; i < Lds::TENSORS; i++) {
            rows[i].measure();
            if (lane == 0) lds.fields(it % Lds::STAGES, my_tensor + i)[slice] = rows[i].field;
        }
    };
    auto commit = [&](int it, auto step) {
        constexpr int i = decltype(step)::value % Lds::TENSORS, share = decltype(step)::value / Lds::TENSORS;
        if constexpr (decltype(step)::value < STEPS)
            rows[i].template commit<share>(lds.tile(it % Lds::STAGES, my_tensor + i), slice * (32 / NSL), lane);
    };
    auto commit_all = [&](int it) {
        if (!fetched) return;
        measure(it);
        static_for<STEPS>([&](auto step) { commit(it, step); });
    };
    fetch(0);
    // LSE2 and delta of the lane's row.  A row that attends to nothing has LSE2 = -inf and only masked entries.
    float lse_q = 0.f, delta_q = 0.f;
    if (n < q_rows) lse_q = p.lse[b * p.lse_b + hd * p.lse_h + q_pos];
    if (p.delta_out != nullptr) {
        // (rows at and beyond lens[b]: the dK/dV launch that follows reads delta of every row of the blocks it visits)
        const float* optr = reinterpret_cast<const float*>(p.o) + b * p.so.b + hd * p.so.h + (int64_t)qb * p.so.t;
        Resident<f32_t, D> raw;
        load_resident<f32_t, D>(raw, doptr, p.sdo.t, q_rows, lane);
        const float d = resident_row_delta<f32_t, D>(raw, optr, p.so.t, q_rows, lane);
        delta_q = qb < seq_len ? d : 0.f;
        if (stream == 0 && h == 0 && n < q_rows) p.delta_out[b * p.delta_b + hd * p.delta_h + q_pos] = delta_q;
    } else if (n < q_rows) {
        delta_q = p.delta[b * p.delta_b + hd * p.delta_h + q_pos];
    }
    ResidentParts<D> qf, dof;
    qf.load(qptr, p.sq.t, q_seen, lane);
    dof.load(doptr, p.sdo.t, q_seen, lane);
    OperandOffsets<f16_t, D> ofs;
    ofs.init(lane);
    commit_all(0);
    fetch(1);

    f32x16 dq[DB];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < DB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) dq[i][r] = 0.f;
    };
    clear();
    const Range vis = visible_range<MASK, true>(q_pos, seq_len, p.margs);
    auto mask = [&](f32x16& pr, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, true>(pr, vis, q_pos, blk * 32, seq_len, p.margs, h, 0.f);
    };

    GradientSum sum;
    for (int it = 0; it < n_iters; it++) {
        if constexpr (R > 1) __syncthreads();  // block `it` is in LDS; everyone is done with the block before
        const int stage = it % Lds::STAGES, blk = hull.lo + it * S + stream;
        const bool mine = blk >= wr.start && blk < wr.end;
        f32x16 s, dp;
        TransposedParts<D, kAhead> kt((const lds_char*)lds.tile(stage, 0), ofs, lane);
        if (mine) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = 0.f;
                dp[r] = 0.f;
            }
            // beside these MFMAs the next block's scale is found, then it is split (one past the end: rows that nobody reads)
            s = mma_rowwise_parts<D>((const lds_char*)lds.tile(stage, 0), ofs, qf, s, lane, [&](auto t) {
                if constexpr (R > 1 && t == 0) measure(it + 1);
            });
            dp = mma_rowwise_parts<D>((const lds_char*)lds.tile(stage, 1), ofs, dof, dp, lane, [&](auto t) {
                constexpr int PER = (STEPS + D / 16 - 1) / (D / 16);
                if constexpr (R > 1) static_for<PER>([&](auto e) { commit(it + 1, std::integral_constant<int, t * PER + e>{}); });
            });
            kt.begin();
        } else if (R > 1) {
            commit_all(it + 1);
        }
        if (R > 1) fetch(it + 2);
        if (mine) {
            int k_field[NSL], v_field[NSL];
            lds.read_fields(stage, 0, k_field);
            lds.read_fields(stage, 1, v_field);
            float f[NSL], g[NSL];
            unscale_factors(k_field, qf.inverse * p.scale_log2, f);
            unscale_factors(v_field, dof.inverse, g);
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = fast_exp2(__builtin_fmaf(s[r], f[(r / 4) * NSL / 4], -lse_q));
            mask(s, blk);
#pragma unroll
            for (int r = 0; r < 16; r++) dp[r] = s[r] * __builtin_fmaf(dp[r], g[(r / 4) * NSL / 4], -delta_q);
            sum.scales(dp, k_field, dq, f);
            kt.run(dp, f, dq);  // dQ^T += K^T dS^T
        }
        if (R == 1) {
            commit_all(it + 1);
            fetch(it + 2);
        }
    }
    sum.finish(dq);
    if (__builtin_amdgcn_ballot_w64(finite_probe(dq, 0.f) != 0.f) != 0) {
        clear();
        for (int blk = hull.lo + stream; blk < wr.end; blk += S) {
            if (blk < wr.start) continue;
            const int k0 = blk * 32;
            f32x16 s = native_rowwise<D>(kptr + k0 * p.sk.t, p.sk.t, seq_len - k0, qptr, p.sq.t, q_seen, lane);
            f32x16 dp = native_rowwise<D>(vptr + k0 * p.sv.t, p.sv.t, seq_len - k0, doptr, p.sdo.t, q_seen, lane);
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = fast_exp2(s[r] * p.scale_log2 - lse_q);
            mask(s, blk);
#pragma unroll
            for (int r = 0; r < 16; r++) dp[r] = s[r] * (dp[r] - delta_q);
            native_transposed<D>(kptr + k0 * p.sk.t, p.sk.t, seq_len - k0, dp, dq, lane);
        }
    }
    const f32x16* const acc[1] = {dq};
    float* const out[1] = {reinterpret_cast<float*>(p.dq) + b * p.sdq.b + hd * p.sdq.h + (int64_t)q_pos * p.sdq.t};
    const float mult[1] = {p.sm_scale};
    f32_store_gradients<D, R, S, 1, Lds::BYTES>(smem, acc, out, mult, wave, lane, n < q_rows, q_pos < seq_len);
}

// ---------------------------------------------------------------- dK, dV
template <int D, int MASK, int R, int S>
__global__ __launch_bounds__(R * S * 64)
__attribute__((amdgpu_waves_per_eu(f32_waves_per_simd(R, R * S, F32Lds<D, R, S, CHILL_PASS_DKDV>::BYTES))))
void dkdv_f32_kernel(BwdParams p, int n_tiles, int n_groups, int has_full_blocks) {
    typedef F32Lds<D, R, S, CHILL_PASS_DKDV> Lds;
    constexpr int DB = (D + 31) / 32, NSL = Lds::SLICES;
    constexpr int kAhead = 2;  // operands of the last products read ahead
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, j;
    if (!work_item(blockIdx.x, p.B * p.H_kv, n_groups, order_of(p), 1, 1, &bh, &j)) return;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H_kv);
    const int hkv = bh % p.H_kv;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int stream = wave % S, member = wave / S;
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const F32Group<MASK, R, S, false> group(j, n_tiles);
    const Range hull = group.hull(seq_len, p.margs);
    // iterations: the S streams' blocks of the hull for every query head of the GQA group in turn (chill_bwd_dkdv.py:156)
    const int per_head = hull.hi > hull.lo ? (hull.hi - hull.lo + S - 1) / S : 0;
    const int n_iters = per_head * p.group;
    const int tile = group.tile(member);
    const int kb0 = 32 * (tile < 0 ? 0 : tile);
    const int k_pos = kb0 + n;
    const int k_rows = tile >= 0 ? p.T - kb0 : 0, k_seen = tile >= 0 ? seq_len - kb0 : 0;  // (of the tensor, of the sequence)
    TileRange wr = {0, 0, 0, 0};
    if (tile >= 0 && kb0 < seq_len) wr = tile_range_rows_discarded<MASK, false>(kb0, 32, 32, seq_len, has_full_blocks != 0, p.margs);

    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h + (int64_t)kb0 * p.sk.t;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h + (int64_t)kb0 * p.sv.t;
    auto q_of = [&](int g) { return reinterpret_cast<const float*>(p.q) + b * p.sq.b + (hkv * p.group + g) * p.sq.h; };
    auto do_of = [&](int g) { return reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + (hkv * p.group + g) * p.sdo.h; };

    const Lds lds = {smem, stream};
    const int slice = member % NSL, my_tensor = R >= 2 ? member / NSL : 0;
    PartStager<D, 32 / NSL> rows[Lds::TENSORS];
    float vec_next = 0.f;
    // the iteration to fetch next, as (query head, blocks of it)
    int next_head = 0, next_it = 0;
    bool fetched = false;
    auto fetch = [&]() {
        const int q0 = 32 * (hull.lo + next_it * S + stream), row0 = q0 + slice * (32 / NSL);
        fetched = next_head < p.group && q0 < 32 * hull.hi;
        if (fetched) {
#pragma unroll
            for (int i = 0; i < Lds::TENSORS; i++) {
                const bool is_do = my_tensor + i == 1;
                rows[i].fetch(is_do ? do_of(next_head) : q_of(next_head), is_do ? p.sdo.t : p.sq.t, row0, seq_len, lane);
            }
            if (member == 0) {
                // LSE2 (lanes 0..31) and delta (lanes 32..63) of the block's rows; rows past the sequence read as zero
                const int hq = hkv * p.group + next_head;
                const float* src = h == 0 ? p.lse + b * p.lse_b + hq * p.lse_h : p.delta + b * p.delta_b + hq * p.delta_h;
                vec_next = q0 + n < seq_len ? src[q0 + n] : 0.f;
            }
        }
        next_it++;
        if (next_it == per_head) {
            next_it = 0;
            next_head++;
        }
    };
    // what was fetched to LDS: first its scale, then the parts, in STEPS shares
    constexpr int STEPS = PartStager<D, 32 / NSL>::STEPS * Lds::TENSORS;
    auto measure = [&](int stage) {
        if (!fetched) return;
#pragma unroll
        for (int i = 0; i < Lds::TENSORS; i++) {
            rows[i].measure();
            if (lane == 0) lds.fields(stage, my_tensor + i)[slice] = rows[i].field;
        }
        if (member == 0) lds.vec(stage)[lane] = vec_next;
    };
    auto commit = [&](int stage, auto step) {
        constexpr int i = decltype(step)::value % Lds::TENSORS, share = decltype(step)::value / Lds::TENSORS;
        if constexpr (decltype(step)::value < STEPS)
            rows[i].template commit<share>(lds.tile(stage, my_tensor + i), slice * (32 / NSL), lane);
    };
    auto commit_all = [&](int stage) {
        if (!fetched) return;
        measure(stage);
        static_for<STEPS>([&](auto step) { commit(stage, step); });
    };
    fetch();
    ResidentParts<D> kf, vf;
    kf.load(kptr, p.sk.t, k_seen, lane);
    vf.load(vptr, p.sv.t, k_seen, lane);
    OperandOffsets<f16_t, D> ofs;
    ofs.init(lane);
    commit_all(0);
    fetch();

    f32x16 dk[DB], dv[DB];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < DB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                dk[i][r] = 0.f;
                dv[i][r] = 0.f;
            }
    };
    clear();
    const Range vis = visible_range<MASK, false>(k_pos, seq_len, p.margs);
    auto mask = [&](f32x16& pr, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, false>(pr, vis, k_pos, blk * 32, seq_len, p.margs, h, 0.f);
    };

    ProbabilitySum dv_sum;
    GradientSum dk_sum;
    int at = 0;  // iteration inside the head
    for (int it = 0; it < n_iters; it++) {
        if constexpr (R > 1) __syncthreads();  // block `it` is in LDS; everyone is done with the block before
        const int stage = it % Lds::STAGES, blk = hull.lo + at * S + stream;
        at = at + 1 == per_head ? 0 : at + 1;
        const bool mine = blk >= wr.start && blk < wr.end;
        const lds_char* q_tile = (const lds_char*)lds.tile(stage, 0);
        const lds_char* do_tile = (const lds_char*)lds.tile(stage, 1);
        f32x16 s, dp;
        if (mine) {
            const int next = (it + 1) % Lds::STAGES;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = 0.f;
                dp[r] = 0.f;
            }
            // beside these MFMAs the next block's scale is found, then it is split (one past the end: rows that nobody reads)
            s = mma_rowwise_parts<D>(q_tile, ofs, kf, s, lane, [&](auto t) {
                if constexpr (R > 1 && t == 0) measure(next);
            });
            dp = mma_rowwise_parts<D>(do_tile, ofs, vf, dp, lane, [&](auto t) {
                constexpr int PER = (STEPS + D / 16 - 1) / (D / 16);
                if constexpr (R > 1) static_for<PER>([&](auto e) { commit(next, std::integral_constant<int, t * PER + e>{}); });
            });
        } else if (R > 1) {
            commit_all((it + 1) % Lds::STAGES);
        }
        if (R > 1) fetch();
        if (mine) {
            int q_field[NSL], do_field[NSL];
            lds.read_fields(stage, 0, q_field);
            lds.read_fields(stage, 1, do_field);
            float f[NSL], g[NSL];
            unscale_factors(q_field, kf.inverse * p.scale_log2, f);
            unscale_factors(do_field, vf.inverse, g);
            const lds_float* vec = (const lds_float*)lds.vec(stage);
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const f32x4 lse4 = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(vec + 8 * g4 + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; e++) s[4 * g4 + e] = fast_exp2(__builtin_fmaf(s[4 * g4 + e], f[g4 * NSL / 4], -lse4[e]));
        }
        mask(s, blk);
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
            const f32x4 del4 = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(vec + 32 + 8 * g4 + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; e++) dp[4 * g4 + e] = s[4 * g4 + e] * __builtin_fmaf(dp[4 * g4 + e], g[g4 * NSL / 4], -del4[e]);
        }
        TransposedParts<D, kAhead> dot(do_tile, ofs, lane), qt(q_tile, ofs, lane);
        dot.begin();
        dv_sum.scales(do_field, dv, f);
        dot.run(s, f, dv);  // dV^T += dO^T P
        qt.begin();
        dk_sum.scales(dp, q_field, dk, f);
        qt.run(dp, f, dk);  // dK^T += Q^T dS
        }
        if (R == 1) {
            commit_all((it + 1) % Lds::STAGES);
            fetch();
        }
    }
    dv_sum.finish(dv);
    dk_sum.finish(dk);
    if (__builtin_amdgcn_ballot_w64(finite_probe(dk, finite_probe(dv, 0.f)) != 0.f) != 0) {
        clear();
        for (int gh = 0; gh < p.group; gh++) {
            const int hq = hkv * p.group + gh;
            const float *lse = p.lse + b * p.lse_b + hq * p.lse_h, *delta = p.delta + b * p.delta_b + hq * p.delta_h;
            for (int blk = hull.lo + stream; blk < wr.end; blk += S) {
                if (blk < wr.start) continue;
                const int q0 = blk * 32;
                const float *qp = q_of(gh) + q0 * p.sq.t, *dop = do_of(gh) + q0 * p.sdo.t;
                f32x16 s = native_rowwise<D>(qp, p.sq.t, seq_len - q0, kptr, p.sk.t, k_seen, lane);
                f32x16 dp = native_rowwise<D>(dop, p.sdo.t, seq_len - q0, vptr, p.sv.t, k_seen, lane);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int q = q0 + 8 * (r / 4) + 4 * h + (r % 4);
                    s[r] = fast_exp2(s[r] * p.scale_log2 - (q < seq_len ? lse[q] : 0.f));
                    dp[r] -= q < seq_len ? delta[q] : 0.f;
                }
                mask(s, blk);
#pragma unroll
                for (int r = 0; r < 16; r++) dp[r] *= s[r];
                native_transposed<D>(dop, p.sdo.t, seq_len - q0, s, dv, lane);
                native_transposed<D>(qp, p.sq.t, seq_len - q0, dp, dk, lane);
            }
        }
    }
    const f32x16* const acc[2] = {dk, dv};
    float* const out[2] = {reinterpret_cast<float*>(p.dk) + b * p.sdk.b + hkv * p.sdk.h + (int64_t)k_pos * p.sdk.t,
                           reinterpret_cast<float*>(p.dv) + b * p.sdv.b + hkv * p.sdv.h + (int64_t)k_pos * p.sdv.t};
    const float mult[2] = {p.sm_scale, 1.f};
    f32_store_gradients<D, R, S, 2, Lds::BYTES>(smem, acc, out, mult, wave, lane, n < k_rows, k_pos < seq_len);
}

// ---------------------------------------------------------------- dK, dV of rows of 512 bytes
// A wave that owns a key tile of such rows would hold K, V and two accumulators of 64 registers each.  Two waves share a tile
// instead: wave 0 holds the K rows and computes P, wave 1 the V rows and dP - delta; they trade the two through LDS, and each
// accumulates half of the head-dim blocks of dV^T and dK^T.  No MFMA is issued twice, both issue the same number; eight waves,
// four tiles, two barriers per 32-query block.  (The same split with fp32 MFMAs, dkdv_split_kernel, which still serves rows of
// 1 KiB: causal B1 H8 T1024 327 us, here 112; full mask B4 H16/4 T1500 1880 and 635.)
template <int D, int MASK>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void dkdv_f32_wide_kernel(BwdParams p, int n_tiles, int n_groups,
                                                                                                     int has_full_blocks) {
    typedef F32Lds<D, 8, 1, CHILL_PASS_DKDV> Lds;
    constexpr int DBW = D / 64, NSL = Lds::SLICES, kAhead = 2;  // head-dim blocks a wave accumulates
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, j;
    if (!work_item(blockIdx.x, p.B * p.H_kv, n_groups, order_of(p), 1, 1, &bh, &j)) return;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H_kv);
    const int hkv = bh % p.H_kv;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int member = wave % 4, role = wave / 4;
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const F32Group<MASK, 4, 1, false> group(j, n_tiles);
    const Range hull = group.hull(seq_len, p.margs);
    const int per_head = hull.hi > hull.lo ? hull.hi - hull.lo : 0;
    const int n_iters = per_head * p.group;  // every query head of the GQA group in turn (chill_bwd_dkdv.py:156)
    const int tile = group.tile(member);
    const int kb0 = 32 * (tile < 0 ? 0 : tile);
    const int k_pos = kb0 + n;
    const int k_rows = tile >= 0 ? p.T - kb0 : 0, k_seen = tile >= 0 ? seq_len - kb0 : 0;  // (of the tensor, of the sequence)
    TileRange wr = {0, 0, 0, 0};
    if (tile >= 0 && kb0 < seq_len) wr = tile_range_rows_discarded<MASK, false>(kb0, 32, 32, seq_len, has_full_blocks != 0, p.margs);

    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h + (int64_t)kb0 * p.sk.t;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h + (int64_t)kb0 * p.sv.t;
    auto q_of = [&](int g) { return reinterpret_cast<const float*>(p.q) + b * p.sq.b + (hkv * p.group + g) * p.sq.h; };
    auto do_of = [&](int g) { return reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + (hkv * p.group + g) * p.sdo.h; };

    // role 0 brings Q, role 1 dO, every wave eight rows
    const Lds lds = {smem, 0};
    PartStager<D, 32 / NSL> rows;
    constexpr int STEPS = PartStager<D, 32 / NSL>::STEPS;
    float vec_next = 0.f;
    int next_head = 0, next_it = 0;
    bool fetched = false;
    auto fetch = [&]() {
        fetched = next_head < p.group && per_head > 0;
        if (!fetched) return;
        const int q0 = 32 * (hull.lo + next_it), row0 = q0 + member * (32 / NSL);
        rows.fetch(role == 1 ? do_of(next_head) : q_of(next_head), role == 1 ? p.sdo.t : p.sq.t, row0, seq_len, lane);
        if (wave == 0) {
            // LSE2 (lanes 0..31) and delta (lanes 32..63) of the block's rows; rows past the sequence read as zero
            const int hq = hkv * p.group + next_head;
            const float* src = h == 0 ? p.lse + b * p.lse_b + hq * p.lse_h : p.delta + b * p.delta_b + hq * p.delta_h;
            vec_next = q0 + n < seq_len ? src[q0 + n] : 0.f;
        }
        next_it++;
        if (next_it == per_head) {
            next_it = 0;
            next_head++;
        }
    };
    auto measure = [&](int stage) {
        if (!fetched) return;
        rows.measure();
        if (lane == 0) lds.fields(stage, role)[member] = rows.field;
        if (wave == 0) lds.vec(stage)[lane] = vec_next;
    };
    auto commit = [&](int stage, auto step) {
        if constexpr (decltype(step)::value < STEPS) rows.template commit<decltype(step)::value>(lds.tile(stage, role), member * (32 / NSL), lane);
    };
    fetch();
    ResidentParts<D> own;
    own.load(role == 1 ? vptr : kptr, role == 1 ? p.sv.t : p.sk.t, k_seen, lane);
    OperandOffsets<f16_t, D> ofs, ofs_tr;  // of all blocks row-wise; of this wave's head-dim blocks transposed
    ofs.init(lane);
#pragma unroll
    for (int i = 0; i < DBW; i++)
#pragma unroll
        for (int w = 0; w < 2; w++) ofs_tr.tr[i][0][w] = role == 0 ? ofs.tr[i][0][w] : ofs.tr[DBW + i][0][w];
    measure(0);
    static_for<STEPS>([&](auto step) { commit(0, step); });
    fetch();

    f32x16 dk[DBW], dv[DBW];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < DBW; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                dk[i][r] = 0.f;
                dv[i][r] = 0.f;
            }
    };
    clear();
    const Range vis = visible_range<MASK, false>(k_pos, seq_len, p.margs);
    auto mask = [&](f32x16& pr, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, false>(pr, vis, k_pos, blk * 32, seq_len, p.margs, h, 0.f);
    };
    f32x4* const give = reinterpret_cast<f32x4*>(smem + f32_wide_ring_bytes(D)) + (member * 2 + role) * 4 * 64 + lane;
    const f32x4* const take = reinterpret_cast<const f32x4*>(smem + f32_wide_ring_bytes(D)) + (member * 2 + 1 - role) * 4 * 64 + lane;

    ProbabilitySum dv_sum;
    GradientSum dk_sum;
    int at = 0;  // iteration inside the head
    for (int it = 0; it < n_iters; it++) {
        __syncthreads();  // block `it` is in LDS; everyone is done with the block before
        const int stage = it & 1, next = stage ^ 1, blk = hull.lo + at;
        at = at + 1 == per_head ? 0 : at + 1;
        const bool mine = blk >= wr.start && blk < wr.end;
        f32x16 x;
        if (mine) {
#pragma unroll
            for (int r = 0; r < 16; r++) x[r] = 0.f;
            x = mma_rowwise_parts<D>((const lds_char*)lds.tile(stage, role), ofs, own, x, lane, [&](auto t) {
                if constexpr (t == 0) measure(next);
            });
            int field[NSL];
            lds.read_fields(stage, role, field);
            float f[NSL];
            unscale_factors(field, role == 0 ? own.inverse * p.scale_log2 : own.inverse, f);
            const lds_float* vec = (const lds_float*)lds.vec(stage) + 32 * role;
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const f32x4 v4 = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(vec + 8 * g4 + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; e++) x[4 * g4 + e] = __builtin_fmaf(x[4 * g4 + e], f[g4 * NSL / 4], -v4[e]);
            }
            if (role == 0) {
#pragma unroll
                for (int r = 0; r < 16; r++) x[r] = fast_exp2(x[r]);
                mask(x, blk);
            }
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) give[r4 * 64] = f32x4{x[4 * r4], x[4 * r4 + 1], x[4 * r4 + 2], x[4 * r4 + 3]};
        } else {
            measure(next);
        }
        __syncthreads();  // P and dP - delta of this block are in LDS
        if (mine) {
            TransposedParts<D, kAhead, DBW> dot((const lds_char*)lds.tile(stage, 1), ofs_tr, lane),
                qt((const lds_char*)lds.tile(stage, 0), ofs_tr, lane);
            dot.begin();
            f32x16 pr, ds;
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
                const f32x4 y = take[r4 * 64];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float a = x[4 * r4 + e], c = y[e];
                    pr[4 * r4 + e] = role == 0 ? a : c;
                    ds[4 * r4 + e] = a * c;
                }
            }
            int q_field[NSL], do_field[NSL];
            lds.read_fields(stage, 0, q_field);
            lds.read_fields(stage, 1, do_field);
            float f[NSL];
            constexpr int PER = (STEPS + 2 * DBW - 1) / (2 * DBW);
            dv_sum.scales(do_field, dv, f);
            dot.run(pr, f, dv, [&](auto u) {  // dV^T += dO^T P
                static_for<PER>([&](auto e) { commit(next, std::integral_constant<int, u * PER + e>{}); });
            });
            qt.begin();
            dk_sum.scales(ds, q_field, dk, f);
            qt.run(ds, f, dk);  // dK^T += Q^T dS
        } else {
            static_for<STEPS>([&](auto step) { commit(next, step); });
        }
        fetch();
    }
    dv_sum.finish(dv);
    dk_sum.finish(dk);
    if (__builtin_amdgcn_ballot_w64(finite_probe(dk, finite_probe(dv, 0.f)) != 0.f) != 0) {
        clear();
        for (int gh = 0; gh < p.group; gh++) {
            const int hq = hkv * p.group + gh;
            const float *lse = p.lse + b * p.lse_b + hq * p.lse_h, *delta = p.delta + b * p.delta_b + hq * p.delta_h;
            for (int blk = wr.start; blk < wr.end; blk++) {
                const int q0 = blk * 32;
                const float *qp = q_of(gh) + q0 * p.sq.t, *dop = do_of(gh) + q0 * p.sdo.t;
                f32x16 s = native_rowwise<D>(qp, p.sq.t, seq_len - q0, kptr, p.sk.t, k_seen, lane);
                f32x16 dp = native_rowwise<D>(dop, p.sdo.t, seq_len - q0, vptr, p.sv.t, k_seen, lane);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int q = q0 + 8 * (r / 4) + 4 * h + (r % 4);
                    s[r] = fast_exp2(s[r] * p.scale_log2 - (q < seq_len ? lse[q] : 0.f));
                    dp[r] -= q < seq_len ? delta[q] : 0.f;
                }
                mask(s, blk);
#pragma unroll
                for (int r = 0; r < 16; r++) dp[r] *= s[r];
                native_transposed<D>(dop, p.sdo.t, seq_len - q0, s, dv, lane, DBW * role);
                native_transposed<D>(qp, p.sq.t, seq_len - q0, dp, dk, lane, DBW * role);
            }
        }
    }
    // lane (n, h) holds columns 32 * (DBW * role + i) + 8 * (r / 4) + 4 * h + r % 4 of ITS key row
    if (n >= k_rows) return;
    const bool valid = k_pos < seq_len;
    float* dkrow = reinterpret_cast<float*>(p.dk) + b * p.sdk.b + hkv * p.sdk.h + (int64_t)k_pos * p.sdk.t + 32 * DBW * role + 4 * h;
    float* dvrow = reinterpret_cast<float*>(p.dv) + b * p.sdv.b + hkv * p.sdv.h + (int64_t)k_pos * p.sdv.t + 32 * DBW * role + 4 * h;
#pragma unroll
    for (int u = 0; u < 4 * DBW; u++) {
        f32x4 a, c;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            a[e] = valid ? dk[u / 4][4 * (u % 4) + e] * p.sm_scale : 0.f;
            c[e] = valid ? dv[u / 4][4 * (u % 4) + e] : 0.f;
        }
        *reinterpret_cast<f32x4*>(dkrow + 8 * u) = a;
        *reinterpret_cast<f32x4*>(dvrow + 8 * u) = c;
    }
}

}  // namespace chill
