// Forward, dQ and dK/dV of fp32 launches that fill the chip, with their matrix products through bf16 parts (chill_f32_parts.h).
//
// A workgroup owns 128 rows of a head (queries in the forward and dQ, keys in dK/dV), 32 a wave, and walks the 32-row blocks of the
// other axis.  Its four waves share the splits of a block: each takes a quarter of the block's rows from global memory into
// registers two blocks ahead, splits it between the matrix instructions of the block before, and leaves the parts in LDS
// (F32Planes), where every wave reads them row by row and transposed.  Two stages, one workgroup barrier a block.  The forward and
// dQ (at head dim 64 with the low parts of dO in LDS) fit in 256 registers, two workgroups a CU; dK/dV at head dim 64, with the parts of
// K and V and two accumulators, takes one wave a SIMD, and so does everything at head dim 128, where the two stages are 96 KiB of LDS:
// 309, 425 and 510 registers in the three kernels.  dK/dV at head dim 16 spills 43 to 53 of 256, all but four of them around what it
// leaves to the fp32 instruction, behind the loop.
// What bounds it: issue.  At head dim 64 a block is 48, 72 and 96 MFMAs of 32 cycles and 330 to 560 vector instructions to a wave, which
// hide behind the MFMAs in part: those are 53, 65 and 47 % of the time (causal B4 H16 T4096, 720 / 942 / 1477 us; the fp32
// instruction's own cycles are 89, 89 and 84 % of its 1119 / 1708 / 2209).  At head dim 128 (the same sizes, 2300 / 3605 / 5325 -> 1549 /
// 2014 / 2727 us) it is 96, 144 and 192 MFMAs, 42, 49 and 48 % of the time at 2.4 GHz: a wave has its SIMD to itself.
#pragma once

#include "chill_device.h"
#include "chill_f32_parts.h"
#include "chill_mask.h"
#include "chill_params.h"
#include "chill_tiles.h"

namespace chill {

constexpr int kF32GroupWaves = 4;

// A thread's share of a block: eight columns of a row of both tensors, at head dims below 64 of one of them (at head dim 16 two
// waves do the same).  Neighbouring lanes take neighbouring columns: whole rows from global memory and to LDS, where an operand's own
// lanes, a row each, met in the banks for 25 cycles a write (causal D64 B4 H16 T4096 728 / 959 / 1495 -> 704 / 936 / 1460 us).
template <int D>
struct F32Share {
    static constexpr int N = D / 16, JOBS = N > 2 ? N / 2 : 1, CHUNKS = D / 8;
    static constexpr int HALVES = JOBS > 2 ? 2 : 1;  // at head dim 128 jobs 2 t and 2 t + 1 are rows 0 .. 15 and 16 .. 31 of a tensor
    typedef F32Planes<D> Planes;
    bool second;        // (JOBS = 1: the wave's tensor)
    int row, col, dst;  // row of the block, first column, their place in the planes of a tensor
    f32x4 x[JOBS][2];
    SplitJob job[JOBS];
    int lost = 0;  // as SplitJob's
    __device__ __forceinline__ void init(int tid) {
        static_assert(JOBS * kF32GroupWaves * 64 >= 2 * 32 * CHUNKS && JOBS <= 4, "a share covers a block");
        const int at = JOBS >= 2 ? tid : tid % (2 * 32 * CHUNKS);
        second = JOBS == 1 && __builtin_amdgcn_readfirstlane(at / (32 * CHUNKS)) != 0;
        row = at % (32 * CHUNKS) / CHUNKS;
        col = 8 * (at % CHUNKS);
        dst = (second ? Planes::BYTES : 0) + Planes::L::chunk_off(row, at % CHUNKS);
    }
    // rows row0 .. row0 + 31 of a and b (rows at and beyond `rows` repeat the last one)
    template <int I>
    __device__ __forceinline__ void load(const float* a, int64_t a_stride, const float* b, int64_t b_stride, int row0, int rows) {
        const bool other = JOBS >= 2 ? I / HALVES == 1 : second;
        const float* src = (other ? b : a) + (int64_t)imin(row0 + row + 16 * (I % HALVES), rows - 1) * (other ? b_stride : a_stride) + col;
        x[I][0] = *reinterpret_cast<const f32x4*>(src);
        x[I][1] = *reinterpret_cast<const f32x4*>(src + 4);
    }
    template <int I>
    __device__ __forceinline__ void take() {
        job[I].x = __builtin_shufflevector(x[I][0], x[I][1], 0, 1, 2, 3, 4, 5, 6, 7);
    }
    template <int I, int PART>
    __device__ __forceinline__ void write(char* stage) const {
        const Parts& p = job[I].p;
        static_assert(HALVES == 1 || OperandOffsets<bf16_t, D>::kHalfAffine, "16 rows further the swizzle is the same");
        constexpr int half = (I % HALVES) * 16 * D * 2;
        *reinterpret_cast<i32x4*>(stage + I / HALVES * Planes::BYTES + PART * Planes::PLANE + half + dst) = PART == 0 ? p.h : PART == 1 ? p.m : p.l;
    }
    template <typename Load>
    __device__ __forceinline__ void at_once(char* stage, Load&& load_next) {
        static_for<JOBS>([&](auto i) {
            take<i>();
            load_next(i);
            job[i].all(lost);
            static_for<3>([&](auto part) { write<i, part>(stage); });
        });
    }
    // slot I of the first phase of a block, which has 6 N
    template <int I, typename Load>
    __device__ __forceinline__ void slot(char* stage, Load&& load_next) {
        constexpr int t = I / 6, part = I % 6;
        if constexpr (t < JOBS) {
            if constexpr (part == 0) take<t>();
            job[t].template share<part>(lost);
            if constexpr (part == 1) load_next(std::integral_constant<int, t>{});
        }
        if constexpr (t > 0 && t <= JOBS && part < 3) write<t - 1, part>(stage);
        if constexpr (I == 6 * N - 1 && N == JOBS) static_for<3>([&](auto k) { write<JOBS - 1, k>(stage); });
    }
};

// Which waves have, among their own blocks, one whose splits lost bits: bit w for wave w, whose 32 rows begin 32 w behind `first`.
// `lost` is a thread's share of block blk.  (what is in the branch runs for values below 2^-109)
template <int MASK, bool QROWS>
struct F32LostBlocks {
    int waves = 0;
    __device__ __forceinline__ void note(int& lost, int blk, int first, int seq_len, MaskArgs a) {
        if (lanes_that_lost(lost) == 0) return;
        lost = 0;
#pragma unroll 1
        for (int w = 0; w < kF32GroupWaves; w++) {
            const TileRange wr = tile_range<MASK, QROWS>(first + 32 * w, 32, 32, seq_len, false, a);
            if (blk >= wr.start && blk < wr.end) waves |= 1 << w;
        }
    }
    // whether this wave is one of them, by what the four have seen (words at 1024 of LDS that nobody reads any more)
    __device__ __forceinline__ bool mine(char* smem, int wave, int lane) const {
        int* words = reinterpret_cast<int*>(smem + 1024);
        if (lane == 0) words[wave] = waves;
        __syncthreads();
        return ((words[0] | words[1] | words[2] | words[3]) >> wave & 1) != 0;
    }
};

template <int D>
__device__ __forceinline__ Parts f32_row_operand(const lds_char* planes, const OperandOffsets<bf16_t, D>& ofs, int j, int lane) {
    typedef F32Planes<D> Planes;
    return Parts{ofs.row_chunk(planes, 0, j, lane), ofs.row_chunk(planes + Planes::PLANE, 0, j, lane), ofs.row_chunk(planes + 2 * Planes::PLANE, 0, j, lane)};
}

template <int N>
__device__ __forceinline__ void clear_f32_blocks(f32x16 (&acc)[N]) {
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
}

// ------------------------------------------------------------------------------------------ forward
template <int D, int MASK>
__global__ __launch_bounds__(kF32GroupWaves * 64) __attribute__((amdgpu_waves_per_eu(D < 64 ? 4 : D < 128 ? 2 : 1))) void fwd_group_f32_kernel(FwdParams p, int n_q_tiles, int has_full_blocks) {
    constexpr int TQ = kF32GroupWaves * 32, NT = kF32GroupWaves * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int STAGE = 2 * Planes::BYTES;  // K, V
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, qt;
    if (!work_item(blockIdx.x, p.B * p.H, n_q_tiles, order_of(p), p.group, f32_group_resident(D, CHILL_PASS_FWD), &bh, &qt)) return;
    qt = n_q_tiles - 1 - qt;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H);
    const int hd = bh % p.H, hkv = hd / p.group;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const int qb = qt * TQ;
    float* obase = reinterpret_cast<float*>(p.o) + b * p.so.b + hd * p.so.h;
    float* lse_base = p.lse ? p.lse + b * p.lse_b + hd * p.lse_h : nullptr;
    if (qb >= seq_len) {
        // nothing attends here: the output rows are defined to be zero (chill.py:96, chill_fwd.py:70-71)
        const int nrows = imin(TQ, p.T - qb);
        zero_rows<f32_t, D, NT>(obase, p.so.t, qb, nrows, tid);
        if (lse_base)
            for (int i = tid; i < nrows; i += NT) lse_base[qb + i] = 0.f;
        return;
    }
    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    // the workgroup's key blocks, and among them the wave's (utils.py:221-272)
    const TileRange wg = tile_range<MASK, true>(qb, TQ, 32, seq_len, false, p.margs);
    const int qw = qb + 32 * wave;
    TileRange wr = tile_range<MASK, true>(qw, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    if (qw >= seq_len) wr.end = wr.start;
    const int last = imax(wg.end - 1, 0);
    F32Share<D> share;
    share.init(tid);
    auto load = [&](auto i, int blk) { share.template load<i>(kptr, p.sk.t, vptr, p.sv.t, imin(blk, last) * 32, seq_len); };
    static_for<F32Share<D>::JOBS>([&](auto i) { load(i, wg.start); });
    F32Resident<D> q;
    uint64_t lost_rows;
    {
        F32Rows<D> rows;
        rows.load_all(F32Rows<D>::at(qptr, p.sq.t, qw, seq_len, lane));
        share.at_once(smem, [&](auto i) { load(i, wg.start + 1); });
        int lost_q = 0;
        q.split(rows, lost_q);
        lost_rows = lanes_that_lost(lost_q);
    }
    F32LostBlocks<MASK, true> lost;
    lost.note(share.lost, wg.start, qb, seq_len, p.margs);
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);

    f32x16 o[DB];
    float m_run = -INFINITY;  // running max of the row (scaled, log2 domain)
    float l_run = 0.f;        // this lane's share of the row sum
    clear_f32_blocks(o);
    const int q_pos = qw + n;
    const Range vis = visible_range<MASK, true>(q_pos, seq_len, p.margs);
    const float scale = p.scale_log2;
    // online softmax (chill_fwd.py:214-226); a row that has seen no key keeps 0 as its reference
    auto softmax = [&](f32x16& s, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, true>(s, vis, q_pos, blk * 32, seq_len, p.margs, h, scale < 0.f ? INFINITY : -INFINITY);
        // (scaled and rounded before the reference is taken off: fused, the rounding of a reference of 1e12 would be the exponent)
        {
#pragma clang fp contract(off)
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = s[r] * scale;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = max_across_halves(mx);
        const float m_new = fmaxf(m_run, mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {
            const float alpha = first_or_rescale(m_run, m_run - m_use);
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[db][r] *= alpha;
            m_run = m_new;
        }
        float psum[2] = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = fast_exp2(s[r] - m_use);
            psum[r % 2] += s[r];
        }
        l_run += psum[0] + psum[1];
    };
    __syncthreads();
    int at = 0;
    for (int blk = wg.start; blk < wg.end; blk++, at ^= 1) {
        const lds_char *k_planes = (const lds_char*)(smem + at * STAGE), *v_planes = k_planes + Planes::BYTES;
        char* next = smem + (at ^ 1) * STAGE;
        auto load_next = [&](auto i) { load(i, blk + 2); };
        if (blk >= wr.start && blk < wr.end) {
            // S^T block: rows = keys 8 * (r / 4) + 4 * h + r % 4 of the block, column n = query row
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            Parts k[2], v[2];
            k[0] = f32_row_operand<D>(k_planes, ofs, 0, lane);
            slots<6 * N>([&](auto i) {
                constexpr int j = i / 6, part = i % 6;
                if constexpr (part == 0 && j + 1 < N) k[(j + 1) % 2] = f32_row_operand<D>(k_planes, ofs, j + 1, lane);
                s = mma_part<part>(k[j % 2], q.p[j], s);
                share.template slot<i>(next, load_next);
            });
            v[0] = Planes::transposed(v_planes, ofs, 0, 0, lane);
            softmax(s, blk);
            SplitJob pj[2];
            pj[0].x = half_of<0>(s) * kPartsUp;
            pj[1].x = half_of<1>(s) * kPartsUp;
            pj[0].all();
            __builtin_amdgcn_sched_barrier(0);
            // O^T += V^T P^T, P scaled up; the second half of P is split beside it
            if constexpr (D == 128) {
                // (a block's share of O added up by itself, as in dQ: the launches of 1024 tiles and more whose keys were shared by four
                // waves had sums a quarter as long.  Full mask B1 H4 T8192 against 64 bits, relative: four sums 7.9e-7, one 14.2e-7, this 3.6e-7)
                static_for<DB>([&](auto db) {
                    f32x16 sum;
#pragma unroll
                    for (int r = 0; r < 16; r++) sum[r] = 0.f;
                    slots<12>([&](auto i) {
                        constexpr int half = i / 6, step = 2 * db + half, part = i % 6;
                        if constexpr (part == 0 && step + 1 < 2 * DB)
                            v[(step + 1) % 2] = Planes::transposed(v_planes, ofs, (step + 1) % 2, (step + 1) / 2, lane);
                        sum = mma_part<part>(v[step % 2], pj[half].p, sum);
                        if constexpr (step == 0) pj[1].template share<part>();
                    });
#pragma unroll
                    for (int r = 0; r < 16; r++) o[db][r] += sum[r];
                });
            } else {
                slots<12 * DB>([&](auto i) {
                    constexpr int step = i / 6, part = i % 6, half = step / DB, db = step % DB;
                    if constexpr (part == 0 && step + 1 < 2 * DB)
                        v[(step + 1) % 2] = Planes::transposed(v_planes, ofs, (step + 1) / DB, (step + 1) % DB, lane);
                    o[db] = mma_part<part>(v[step % 2], pj[half].p, o[db]);
                    if constexpr (step == 0) pj[1].template share<part>();
                });
            }
        } else {
            share.at_once(next, load_next);
        }
        lost.note(share.lost, imin(blk + 1, last), qb, seq_len, p.margs);
        __syncthreads();
    }

    // LSE2 = m + log2(l) (chill_fwd.py:288-289); -inf for a row that saw no key, 0 for rows past lens
    auto store = [&](bool mine) {
        const float l_all = sum_across_halves(l_run), l_safe = (l_all == 0.f) ? 1.f : l_all;
        if (!mine || q_pos >= p.T) return;
        const bool valid = q_pos < seq_len;
        store_row_transposed<f32_t, D>(obase + (int64_t)q_pos * p.so.t, o, 1.f / l_safe, valid, h);
        if (lse_base != nullptr && h == 0) lse_base[q_pos] = valid ? m_run + __log2f(l_safe) : 0.f;
    };
    scale_f32_blocks(o, kPartsDown);
    store(true);
    const float bad = nan_if_not_finite(o, l_run);
    const bool again = lost.mine(smem, wave, lane) || row_that_lost(lost_rows, lane) || bad != bad;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear_f32_blocks(o);
        m_run = -INFINITY;
        l_run = 0.f;
        for (int blk = wr.start; blk < wr.end; blk++) {
            const int k0 = blk * 32;
            f32x16 s = native_rowwise<D>(kptr + (int64_t)k0 * p.sk.t, p.sk.t, seq_len - k0, qptr + (int64_t)qw * p.sq.t, p.sq.t, seq_len - qw, lane);
            softmax(s, blk);
            native_transposed<D>(vptr + (int64_t)k0 * p.sv.t, p.sv.t, seq_len - k0, s, o, lane);
        }
        store(again);
    }
}

// ------------------------------------------------------------------------------------------ dQ
template <int D, int MASK>
__global__ __launch_bounds__(kF32GroupWaves * 64) __attribute__((amdgpu_waves_per_eu(D < 128 ? 2 : 1))) void dq_group_f32_kernel(BwdParams p, int n_q_tiles, int has_full_blocks) {
    constexpr int TQ = kF32GroupWaves * 32, NT = kF32GroupWaves * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int STAGE = 2 * Planes::BYTES;  // K, V
    // Two waves a SIMD have 256 registers each, too few at head dim 64: the low parts of the wave's dO lie in LDS, behind the stages
    // (5 to 7 registers were spilled in the loop
    // otherwise; causal B8 H32 T300 49.5 -> 45.5 us, B32 H32 T128 52.1 -> 47.6, window 100 + 30 B8 H32 T800 127 -> 119, B4 H16 T4096 equal)
    constexpr bool kParked = f32_group_parks(D);
    constexpr int PARKED = 64 * 16;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int bh, qt;
    if (!work_item(blockIdx.x, p.B * p.H, n_q_tiles, order_of(p), p.group, f32_group_resident(D, CHILL_PASS_DQ), &bh, &qt)) return;
    qt = n_q_tiles - 1 - qt;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H);
    const int hd = bh % p.H, hkv = hd / p.group;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const int qb = qt * TQ;
    float* dqbase = reinterpret_cast<float*>(p.dq) + b * p.sdq.b + hd * p.sdq.h;
    if (qb >= seq_len) {
        // rows at or beyond lens[b] receive 0 (the reference relies on the adapter's zero-fill, chill.py:292)
        const int nrows = imin(TQ, p.T - qb);
        zero_rows<f32_t, D, NT>(dqbase, p.sdq.t, qb, nrows, tid);
        // (the dK/dV launch that follows reads delta of every row of the tiles it visits)
        if (p.delta_out != nullptr)
            for (int i = tid; i < nrows; i += NT) p.delta_out[b * p.delta_b + hd * p.delta_h + qb + i] = 0.f;
        return;
    }
    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h;
    const float* doptr = reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hd * p.sdo.h;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    // the workgroup's key blocks, and among them the wave's (utils.py:221-272)
    const TileRange wg = tile_range<MASK, true>(qb, TQ, 32, seq_len, false, p.margs);
    const int qw = qb + 32 * wave;
    TileRange wr = tile_range<MASK, true>(qw, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    if (qw >= seq_len) wr.end = wr.start;
    const int last = imax(wg.end - 1, 0);
    F32Share<D> share;
    share.init(tid);
    auto load = [&](auto i, int blk) { share.template load<i>(kptr, p.sk.t, vptr, p.sv.t, imin(blk, last) * 32, seq_len); };
    static_for<F32Share<D>::JOBS>([&](auto i) { load(i, wg.start); });
    const int q_pos = qw + n;
    F32Resident<D> q, d_o;
    float lse_q = 0.f, delta_q = 0.f;
    uint64_t lost_rows;
    {
        F32Rows<D> rows;
        rows.load_all(F32Rows<D>::at(doptr, p.sdo.t, qw, seq_len, lane));
        if (q_pos < p.T) lse_q = p.lse[b * p.lse_b + hd * p.lse_h + q_pos];
        if (p.delta_out != nullptr) {
            // delta = rowsum(O * dO), 0 for rows past the sequence
            F32Rows<D> out;
            const float* optr = reinterpret_cast<const float*>(p.o) + b * p.so.b + hd * p.so.h;
            out.load_all(F32Rows<D>::at(optr, p.so.t, qw, seq_len, lane));
#pragma unroll
            for (int i = 0; i < 2 * N; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) delta_q += out.c[i][e] * rows.c[i][e];
            delta_q += __shfl_xor(delta_q, 32, 64);
            if (q_pos >= seq_len) delta_q = 0.f;
            if (h == 0 && q_pos < p.T) p.delta_out[b * p.delta_b + hd * p.delta_h + q_pos] = delta_q;
        } else if (q_pos < p.T) {
            delta_q = p.delta[b * p.delta_b + hd * p.delta_h + q_pos];
        }
        d_o.split_scaled_up(rows);
        rows.load_all(F32Rows<D>::at(qptr, p.sq.t, qw, seq_len, lane));
        share.at_once(smem, [&](auto i) { load(i, wg.start + 1); });
        int lost_q = 0;
        q.split(rows, lost_q);
        lost_rows = lanes_that_lost(lost_q);
    }
    F32LostBlocks<MASK, true> lost;
    lost.note(share.lost, wg.start, qb, seq_len, p.margs);
    // a row that attends to nothing has LSE2 = -inf and only masked entries (score -inf): P = exp2(-inf - 0)
    if (lse_q == -INFINITY) lse_q = 0.f;
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);
    char* parked = smem + 2 * STAGE + wave * N * PARKED + lane * 16;
    if constexpr (kParked) static_for<N>([&](auto j) { *reinterpret_cast<i32x4*>(parked + j * PARKED) = d_o.p[j].l; });

    f32x16 dq[DB];
    clear_f32_blocks(dq);
    const Range vis = visible_range<MASK, true>(q_pos, seq_len, p.margs);
    const float scale = p.scale_log2;
    const float masked_score = scale < 0.f ? INFINITY : -INFINITY;  // times the scale: -inf
    auto mask = [&](f32x16& s, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, true>(s, vis, q_pos, blk * 32, seq_len, p.margs, h, masked_score);
    };
    __syncthreads();
    int at = 0;
    for (int blk = wg.start; blk < wg.end; blk++, at ^= 1) {
        const lds_char *k_planes = (const lds_char*)(smem + at * STAGE), *v_planes = k_planes + Planes::BYTES;
        char* next = smem + (at ^ 1) * STAGE;
        auto load_next = [&](auto i) { load(i, blk + 2); };
        if (blk >= wr.start && blk < wr.end) {
            f32x16 s, dp;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = 0.f;
                dp[r] = -delta_q * kPartsUp;
            }
            // S^T and, scaled up, dP^T blocks: rows = keys 8 * (r / 4) + 4 * h + r % 4 of the block, column n = query row
            Parts x[2];
            x[0] = f32_row_operand<D>(k_planes, ofs, 0, lane);
            auto operand = [&](auto t) { x[t % 2] = f32_row_operand<D>(t < N ? k_planes : v_planes, ofs, t % N, lane); };
            i32x4 low;
            auto low_of = [&](auto j) { low = *reinterpret_cast<const lds_i32x4*>((const lds_char*)parked + j * PARKED); };
            slots<6 * N>([&](auto i) {
                constexpr int t = i / 6, part = i % 6;
                if constexpr (part == 0) operand(std::integral_constant<int, t + 1>{});
                s = mma_part<part>(x[t % 2], q.p[t], s);
                share.template slot<i>(next, load_next);
                if constexpr (kParked && i == 6 * N - 4) low_of(std::integral_constant<int, 0>{});
            });
            mask(s, blk);
            constexpr int PER = (16 + 6 * N - 1) / (6 * N);  // exponentials a slot
            slots<6 * N>([&](auto i) {
                constexpr int t = N + i / 6, part = i % 6;
                if constexpr (part == 0) {
                    if constexpr (t + 1 < 2 * N)
                        operand(std::integral_constant<int, t + 1>{});
                    else
                        x[(t + 1) % 2] = Planes::transposed(k_planes, ofs, 0, 0, lane);
                }
                if constexpr (kParked)
                    dp = mma_part<part>(x[t % 2], Parts{d_o.p[t - N].h, d_o.p[t - N].m, low}, dp);
                else
                    dp = mma_part<part>(x[t % 2], d_o.p[t - N], dp);
                if constexpr (kParked && part == 2 && t + 1 < 2 * N) low_of(std::integral_constant<int, t + 1 - N>{});
#pragma unroll
                for (int r = PER * i; r < PER * (i + 1) && r < 16; r++) s[r] = f32_probability(s[r], scale, lse_q);
            });
#pragma unroll
            for (int r = 0; r < 16; r++) dp[r] *= s[r];
            SplitJob job[2];
            job[0].x = half_of<0>(dp);
            job[0].all();
            job[1].x = half_of<1>(dp);
            __builtin_amdgcn_sched_barrier(0);
            // dQ^T += K^T dS^T; the second half of dS is split beside the first one's products.  A block's share of a sum is added up by
            // itself: one rounding of the long sum a block and not twelve
            static_for<DB>([&](auto db) {
                f32x16 sum;
#pragma unroll
                for (int r = 0; r < 16; r++) sum[r] = 0.f;
                slots<12>([&](auto i) {
                    constexpr int half = i / 6, step = 2 * db + half, part = i % 6;
                    if constexpr (part == 0 && step + 1 < 2 * DB)
                        x[(step + 1) % 2] = Planes::transposed(k_planes, ofs, (step + 1) % 2, (step + 1) / 2, lane);
                    sum = mma_part<part>(x[step % 2], job[half].p, sum);
                    if constexpr (step == 0) job[1].template share<part>();
                });
#pragma unroll
                for (int r = 0; r < 16; r++) dq[db][r] += sum[r];
            });
        } else {
            share.at_once(next, load_next);
        }
        lost.note(share.lost, imin(blk + 1, last), qb, seq_len, p.margs);
        __syncthreads();
    }

    auto store = [&](bool mine) {
        if (mine && q_pos < p.T) store_row_transposed<f32_t, D>(dqbase + (int64_t)q_pos * p.sdq.t, dq, p.sm_scale, q_pos < seq_len, h);
    };
    scale_f32_blocks(dq, kPartsDown);
    store(true);
    const float bad = nan_if_not_finite(dq);
    const bool again = lost.mine(smem, wave, lane) || row_that_lost(lost_rows, lane) || bad != bad;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear_f32_blocks(dq);
        for (int blk = wr.start; blk < wr.end; blk++) {
            const int k0 = blk * 32;
            const float *kb = kptr + (int64_t)k0 * p.sk.t, *vb = vptr + (int64_t)k0 * p.sv.t;
            f32x16 s = native_rowwise<D>(kb, p.sk.t, seq_len - k0, qptr + (int64_t)qw * p.sq.t, p.sq.t, seq_len - qw, lane);
            f32x16 dp = native_rowwise<D>(vb, p.sv.t, seq_len - k0, doptr + (int64_t)qw * p.sdo.t, p.sdo.t, seq_len - qw, lane);
            mask(s, blk);
#pragma unroll
            for (int r = 0; r < 16; r++) dp[r] = f32_probability(s[r], scale, lse_q) * (dp[r] - delta_q);
            native_transposed<D>(kb, p.sk.t, seq_len - k0, dp, dq, lane);
        }
        store(again);
    }
}

// ------------------------------------------------------------------------------------------ dK, dV
template <int D, int MASK>
__global__ __launch_bounds__(kF32GroupWaves * 64) __attribute__((amdgpu_waves_per_eu(D < 64 ? 2 : 1))) void dkdv_group_f32_kernel(BwdParams p, int n_k_tiles, int has_full_blocks) {
    constexpr int TK = kF32GroupWaves * 32, NT = kF32GroupWaves * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int VECS = 2 * Planes::BYTES, STAGE = VECS + 2 * 32 * 4;  // Q, dO; LSE2 and -delta of their rows
    extern __shared__ __attribute__((aligned(16))) char smem[];
    // key tiles first-to-last: for causal-like masks the longest run first
    int bh, ktile;
    if (!work_item(blockIdx.x, p.B * p.H_kv, n_k_tiles, order_of(p), 1, f32_group_resident(D, CHILL_PASS_DKDV), &bh, &ktile)) return;
    const int b = batch_by_length(p.lens, p.lens_stride, p.B, p.T, bh / p.H_kv);
    const int hkv = bh % p.H_kv;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const int kb0 = ktile * TK;
    float* dkbase = reinterpret_cast<float*>(p.dk) + b * p.sdk.b + hkv * p.sdk.h;
    float* dvbase = reinterpret_cast<float*>(p.dv) + b * p.sdv.b + hkv * p.sdv.h;
    if (kb0 >= seq_len) {
        // rows at or beyond lens[b] receive 0 (the reference relies on the adapter's zero-fill, chill.py:293-294)
        const int nrows = imin(TK, p.T - kb0);
        zero_rows<f32_t, D, NT>(dkbase, p.sdk.t, kb0, nrows, tid);
        zero_rows<f32_t, D, NT>(dvbase, p.sdv.t, kb0, nrows, tid);
        return;
    }
    // the workgroup's query blocks, and among them the wave's
    const TileRange wg = tile_range<MASK, false>(kb0, TK, 32, seq_len, false, p.margs);
    const int kw = kb0 + 32 * wave;
    TileRange wr = tile_range<MASK, false>(kw, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    if (kw >= seq_len) wr.end = wr.start;
    const int n_blocks = imax(wg.end - wg.start, 0);
    const int n_iters = n_blocks * p.group;  // every query head of the GQA group in turn (chill_bwd_dkdv.py:156)

    const float* q0 = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hkv * p.group * p.sq.h;
    const float* do0 = reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hkv * p.group * p.sdo.h;
    const float* vec0 = h == 0 ? p.lse + b * p.lse_b + hkv * p.group * p.lse_h : p.delta + b * p.delta_b + hkv * p.group * p.delta_h;
    const int64_t vec_head = h == 0 ? p.lse_h : p.delta_h;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;
    // the block whose rows are loaded next (the last one stays): group head, first row
    int ahead = 0, head_ahead = 0, blk_ahead = wg.start;
    auto advance = [&]() {
        if (ahead + 1 >= n_iters) return;
        ahead++;
        if (++blk_ahead >= wg.end) {
            blk_ahead = wg.start;
            head_ahead++;
        }
    };
    F32Share<D> share;
    share.init(tid);
    auto load = [&](auto i) {
        share.template load<i>(q0 + head_ahead * p.sq.h, p.sq.t, do0 + head_ahead * p.sdo.h, p.sdo.t, blk_ahead * 32, seq_len);
    };
    // LSE2 (lanes 0..31) and delta (lanes 32..63) of the block's rows, through LDS (a row that attends to nothing has LSE2 = -inf and
    // only masked entries)
    auto row_vec = [&]() { return vec0[head_ahead * vec_head + imin(blk_ahead * 32 + n, seq_len - 1)]; };
    auto leave_vec = [&](char* stage, float x) {
        reinterpret_cast<float*>(stage + VECS)[lane] = h == 0 ? (x == -INFINITY ? 0.f : x) : -x;
    };
    auto read_vec = [&](const char* stage, int at) {
        f32x16 x;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const f32x4 y = *reinterpret_cast<const f32x4*>(stage + VECS + (at + 8 * g + 4 * h) * 4);
#pragma unroll
            for (int e = 0; e < 4; e++) x[4 * g + e] = y[e];
        }
        return x;
    };
    F32Resident<D> k, v;
    float vec_next = 0.f;
    uint64_t lost_rows = 0;
    F32LostBlocks<MASK, false> lost;
    if (n_iters > 0) {
        static_for<F32Share<D>::JOBS>([&](auto i) { load(i); });
        vec_next = row_vec();
        F32Rows<D> kr, vr;
        kr.load_all(F32Rows<D>::at(kptr, p.sk.t, kw, seq_len, lane));
        vr.load_all(F32Rows<D>::at(vptr, p.sv.t, kw, seq_len, lane));
        if (wave == 0) leave_vec(smem, vec_next);
        advance();
        vec_next = row_vec();
        share.at_once(smem, [&](auto i) { load(i); });
        int lost_kv = 0;
        k.split(kr, lost_kv);
        v.split(vr, lost_kv);
        lost_rows = lanes_that_lost(lost_kv);
        lost.note(share.lost, wg.start, kb0, seq_len, p.margs);
    }
    const int k_pos = kw + n;
    const Range vis = visible_range<MASK, false>(k_pos, seq_len, p.margs);
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);

    f32x16 dk[DB], dv[DB];
    clear_f32_blocks(dk);
    clear_f32_blocks(dv);
    const float scale = p.scale_log2;
    const float masked_score = scale < 0.f ? INFINITY : -INFINITY;  // times the scale: -inf
    auto mask = [&](f32x16& s, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, false>(s, vis, k_pos, blk * 32, seq_len, p.margs, h, masked_score);
    };
    __syncthreads();
    int at = 0, blk = wg.start;
    for (int it = 0; it < n_iters; it++, at ^= 1) {
        char *stage = smem + at * STAGE, *next = smem + (at ^ 1) * STAGE;
        const lds_char *q_planes = (const lds_char*)stage, *do_planes = q_planes + Planes::BYTES;
        if (wave == 0) leave_vec(next, vec_next);
        advance();
        vec_next = row_vec();
        if (blk >= wr.start && blk < wr.end) {
            f32x16 s, dp = read_vec(stage, 32);  // (the dP chain starts from -delta)
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.f;
            // S and dP blocks: rows = queries 8 * (r / 4) + 4 * h + r % 4 of the block, column n = key (the scores with the rounding of
            // the forward's, which LSE2 has: P of a row's largest is then as close to 1 as it was there)
            Parts x[2];
            x[0] = f32_row_operand<D>(q_planes, ofs, 0, lane);
            auto operand = [&](auto t) { x[t % 2] = f32_row_operand<D>(t < N ? q_planes : do_planes, ofs, t % N, lane); };
            slots<6 * N>([&](auto i) {
                constexpr int t = i / 6, part = i % 6;
                if constexpr (part == 0) operand(std::integral_constant<int, t + 1>{});
                s = mma_part_transposed<part>(x[t % 2], k.p[t], s);
                share.template slot<i>(next, load);
            });
            const f32x16 lse = read_vec(stage, 0);
            mask(s, blk);
            // the exponentials (P, and with it dS, scaled up) of the first half of P in the first half of the dP chain, so that it can be split in the last step
            SplitJob pj[2];
            constexpr int PER = (16 + 6 * N - 7) / (6 * N - 6 > 0 ? 6 * N - 6 : 1);
            slots<6 * N>([&](auto i) {
                constexpr int t = N + i / 6, part = i % 6;
                if constexpr (part == 0) {
                    if constexpr (t + 1 < 2 * N)
                        operand(std::integral_constant<int, t + 1>{});
                    else
                        x[(t + 1) % 2] = Planes::transposed(do_planes, ofs, 0, 0, lane);
                }
                dp = mma_part<part>(x[t % 2], v.p[t - N], dp);
                if constexpr (N > 1) {
#pragma unroll
                    for (int r = PER * i; r < PER * (i + 1) && r < 16; r++) s[r] = f32_probability(s[r], scale, lse[r]) * kPartsUp;
                    if constexpr (i == 6 * N - 6) pj[0].x = half_of<0>(s);
                    if constexpr (i >= 6 * N - 6) pj[0].template share<i % 6>();
                }
            });
            if constexpr (N == 1) {
#pragma unroll
                for (int r = 0; r < 16; r++) s[r] = f32_probability(s[r], scale, lse[r]) * kPartsUp;
                pj[0].x = half_of<0>(s);
                pj[0].all();
            }
            pj[1].x = half_of<1>(s);
            __builtin_amdgcn_sched_barrier(0);
            // dV^T += dO^T P, then dK^T += Q^T dS; step w of 4 DB.  Beside them: the second half of P, dS and its two halves.  A block's
            // share of a sum is added up by itself: one rounding of the long sum a block and not twelve
            f32x16 part_sum[2];
            slots<24 * DB>([&](auto i) {
                constexpr int w = i / 6, part = i % 6, half = w % 2, sum = w / 2;
                if constexpr (part == 0 && w + 1 < 4 * DB)
                    x[(w + 1) % 2] = Planes::transposed(w + 1 < 2 * DB ? do_planes : q_planes, ofs, (w + 1) % 2, (w + 1) / 2 % DB, lane);
                if constexpr (part == 0 && half == 0) {
#pragma unroll
                    for (int r = 0; r < 16; r++) part_sum[sum % 2][r] = 0.f;
                }
                part_sum[sum % 2] = mma_part<part>(x[w % 2], pj[half].p, part_sum[sum % 2]);
                if constexpr (half == 0 && sum > 0) {
                    constexpr int before = sum - 1;
                    f32x16& acc = before < DB ? dv[before % DB] : dk[before % DB];
#pragma unroll
                    for (int r = 3 * part; r < 3 * part + 3 && r < 16; r++) acc[r] += part_sum[before % 2][r];
                }
                if constexpr (w == 0) {
                    pj[1].template share<part>();
#pragma unroll
                    for (int r = 3 * part; r < 3 * part + 3 && r < 16; r++) dp[r] *= s[r];
                }
                // (pj[0] is free behind the last but one of dV's steps, pj[1] behind the last)
                if constexpr (w == 2 * DB - 1) {
                    if constexpr (part == 0) pj[0].x = half_of<0>(dp);
                    pj[0].template share<part>();
                }
                if constexpr (w == 2 * DB) {
                    if constexpr (part == 0) pj[1].x = half_of<1>(dp);
                    pj[1].template share<part>();
                }
            });
#pragma unroll
            for (int r = 0; r < 16; r++) dk[DB - 1][r] += part_sum[(2 * DB - 1) % 2][r];
        } else {
            share.at_once(next, load);
        }
        if (++blk >= wg.end) blk = wg.start;
        if (it + 1 < n_iters) lost.note(share.lost, blk, kb0, seq_len, p.margs);
        __syncthreads();
    }

    auto store = [&](bool mine) {
        if (!mine || k_pos >= p.T) return;
        store_row_transposed<f32_t, D>(dkbase + (int64_t)k_pos * p.sdk.t, dk, p.sm_scale, k_pos < seq_len, h);
        store_row_transposed<f32_t, D>(dvbase + (int64_t)k_pos * p.sdv.t, dv, 1.f, k_pos < seq_len, h);
    };
    scale_f32_blocks(dk, kPartsDown);
    scale_f32_blocks(dv, kPartsDown);
    store(true);
    const float bad = nan_if_not_finite(dk, nan_if_not_finite(dv));
    const bool again = lost.mine(smem, wave, lane) || row_that_lost(lost_rows, lane) || bad != bad;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear_f32_blocks(dk);
        clear_f32_blocks(dv);
        char* mine = smem + wave * (2 * 32 * 4) - VECS;  // (leave_vec and read_vec add VECS)
        const float *kb = kptr + (int64_t)kw * p.sk.t, *vb = vptr + (int64_t)kw * p.sv.t;
        for (head_ahead = 0; head_ahead < p.group; head_ahead++) {
            for (blk_ahead = wr.start; blk_ahead < wr.end; blk_ahead++) {
                const int row0 = blk_ahead * 32;
                const float *qb = q0 + head_ahead * p.sq.h + (int64_t)row0 * p.sq.t, *dob = do0 + head_ahead * p.sdo.h + (int64_t)row0 * p.sdo.t;
                leave_vec(mine, row_vec());
                f32x16 s = native_rowwise<D>(qb, p.sq.t, seq_len - row0, kb, p.sk.t, seq_len - kw, lane);
                f32x16 dp = native_rowwise<D>(dob, p.sdo.t, seq_len - row0, vb, p.sv.t, seq_len - kw, lane);
                const f32x16 lse = read_vec(mine, 0), neg_delta = read_vec(mine, 32);
                mask(s, blk_ahead);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    s[r] = f32_probability(s[r], scale, lse[r]);
                    dp[r] = s[r] * (dp[r] + neg_delta[r]);
                }
                native_transposed<D>(dob, p.sdo.t, seq_len - row0, s, dv, lane);
                native_transposed<D>(qb, p.sq.t, seq_len - row0, dp, dk, lane);
            }
        }
        store(again);
    }
}

}  // namespace chill
