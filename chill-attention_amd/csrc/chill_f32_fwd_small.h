// Forward, dQ and dK/dV of fp32 launches with few 32-row tiles: the kernels of chill_fwd_small.h and chill_bwd_small.h, with their
// matrix products through bf16 parts (chill_f32_parts.h).
//
// A workgroup owns one 32-row tile of a head (queries in the forward and dQ, keys in dK/dV) and its waves take the 32-row blocks
// of the other axis in turn, each with accumulators of its own, merged through LDS at the end.  A wave is on its own until then:
// it loads the rows of a block from global memory straight into the registers the split starts from, one block ahead, leaves the
// parts of what is needed transposed as well in LDS (F32Planes), and reads them back with ds_read_b64_tr_b16.  A block is a
// sequence of MFMAs, each followed by its share of the vector work (slots): the split of the operand that is due next, the
// exponentials, the split of P and dS.
#pragma once

#include "chill_f32_parts.h"
#include "chill_fwd_small.h"

namespace chill {

// (TILES and SETS as in fwd_small_kernel; at head dim 16 four waves a SIMD, 128 registers: with three, which the compiler would take,
// causal B4 H8 T1100 is 29 us instead of 24)
template <int D, int MASK, int TILES, int SETS>
__global__ __launch_bounds__(kFwdSmallWaves * 64 * TILES * SETS) __attribute__((amdgpu_waves_per_eu(D < 32 ? 4 : D < 128 ? 2 : 1))) void fwd_small_f32_kernel(FwdParams p, int n_q_tiles, int total_items, int has_full_blocks) {
    constexpr int NW = kFwdSmallWaves * SETS, NT = NW * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int WAVE_BYTES = fwd_small_wave_bytes(D, CHILL_F32);
    extern __shared__ __attribute__((aligned(16))) char smem_all[];
    const int item = blockIdx.x;
    if (item >= total_items) return;
    const int half = TILES == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;  // which q-tile of the workgroup
    char* smem = smem_all + half * (NW * WAVE_BYTES);
    // the q-tiles of all heads from the last to the first (under causal-like masks: longest first)
    const int per_head = TILES == 2 ? (n_q_tiles + 1) / 2 : n_q_tiles;
    const int n_heads = total_items / per_head;
    const int bh = item % n_heads, j = item / n_heads;
    const int qt = half == 0 ? n_q_tiles - 1 - j : j;
    const bool has_tile = half == 0 || n_q_tiles - 1 - j != j;  // (an odd number: the middle one has no partner)
    const int b = bh / p.H, hd = bh % p.H, hkv = hd / p.group;
    const int tid = threadIdx.x % NT, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const int qb = qt * 32;
    float* obase = reinterpret_cast<float*>(p.o) + b * p.so.b + hd * p.so.h;
    float* lse_base = p.lse ? p.lse + b * p.lse_b + hd * p.lse_h : nullptr;
    if (!has_tile || qb >= seq_len) {
        if (has_tile) {
            // nothing attends here: the output rows are defined to be zero (chill.py:96, chill_fwd.py:70-71)
            const int nrows = imin(32, p.T - qb);
            zero_rows<f32_t, D, NT>(obase, p.so.t, qb, nrows, tid);
            if (lse_base)
                for (int i = tid; i < nrows; i += NT) lse_base[qb + i] = 0.f;
        }
        if constexpr (TILES == 2) __syncthreads();  // the other half's one barrier
        return;
    }
    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    // the 32-key blocks of these rows (utils.py:221-272 with 32 x 32 tiles)
    const TileRange wr = tile_range<MASK, true>(qb, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    const int first = wr.start + wave;
    F32Rows<D> k, v;
    F32Resident<D> q;
    int lost = 0;  // (of K and V)
    uint64_t lost_rows;
    {
        F32Rows<D> rows;
        rows.load_all(F32Rows<D>::at(qptr, p.sq.t, qb, seq_len, lane));
        const int blk = imax(imin(first, wr.end - 1), 0);  // (a wave without blocks loads one all the same)
        k.load_all(F32Rows<D>::at(kptr, p.sk.t, blk * 32, seq_len, lane));
        v.load_all(F32Rows<D>::at(vptr, p.sv.t, blk * 32, seq_len, lane));
        int lost_q = 0;
        q.split(rows, lost_q);
        lost_rows = lanes_that_lost(lost_q);
    }
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);
    char* mine = smem + wave * WAVE_BYTES;
    const lds_char* planes = (const lds_char*)mine;

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
    const int q_pos = qb + n;
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

    SplitJob kj[N];  // K of the block that is due
    static_for<N>([&](auto j) {
        kj[j].x = k.template operand<j>();
        kj[j].all(lost);
    });
    for (int blk = first; blk < wr.end; blk += NW) {
        const int next = blk + NW < wr.end ? blk + NW : blk;
        const float* k_next = F32Rows<D>::at(kptr, p.sk.t, next * 32, seq_len, lane);
        const float* v_next = F32Rows<D>::at(vptr, p.sv.t, next * 32, seq_len, lane);
        if constexpr (D < 128) k.load_all(k_next);
        // S^T block: rows = keys 8 * (r / 4) + 4 * h + r % 4 of the block, column n = query row; V is split beside it
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.f;
        SplitJob vj[2];
        slots<6 * N>([&](auto i) {
            constexpr int j = i / 6, part = i % 6;
            s = mma_part<part>(kj[j].p, q.p[j], s);
            if constexpr (part == 0) vj[j % 2].x = v.template operand<j>();
            vj[j % 2].template share<part>(lost);
            if constexpr (part == 2) v.template load<j>(v_next);
            // (at head dim 128 into the registers of the operand that was due: no register is spilled, where 8 were under a causal mask, and
            // a band of 256 + 256 took three times as long)
            if constexpr (D == 128 && part == 5) k.template load<j>(k_next);
            if constexpr (j > 0 && part < 3) Planes::template write<j - 1, part>(mine, vj[(j + 1) % 2].p, lane);
        });
        static_for<3>([&](auto part) { Planes::template write<N - 1, part>(mine, vj[(N - 1) % 2].p, lane); });
        Parts vt[2];
        vt[0] = Planes::transposed(planes, ofs, 0, 0, lane);
        softmax(s, blk);
        SplitJob pj[2];
        pj[0].x = half_of<0>(s) * kPartsUp;
        pj[1].x = half_of<1>(s) * kPartsUp;
        pj[0].all();
        __builtin_amdgcn_sched_barrier(0);
        // O^T += V^T P^T, P scaled up; the second half of P and the next block's K are split beside it
        slots<12 * DB>([&](auto i) {
            constexpr int step = i / 6, part = i % 6, half = step / DB, db = step % DB;
            o[db] = mma_part<part>(vt[step % 2], pj[half].p, o[db]);
            if constexpr (part == 0 && step + 1 < 2 * DB)
                vt[(step + 1) % 2] = Planes::transposed(planes, ofs, (step + 1) / DB, (step + 1) % DB, lane);
            if constexpr (step == 0) pj[1].template share<part>();
            // (N = 2 DB operands at head dims from 32 on: one a step)
            constexpr int j = step;
            if constexpr (j < N) {
                if constexpr (part == 0) kj[j].x = k.template operand<j>();
                kj[j].template share<part>(lost);
            }
        });
    }
    scale_f32_blocks(o, kPartsDown);
    fwd_small_leave<DB>(mine, WAVE_BYTES, lane, o, m_run, sum_across_halves(l_run));
    const float bad = nan_if_not_finite(o, l_run);
    const bool again = bad != bad || row_that_lost(lost_rows, lane) || lanes_that_lost(lost) != 0;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear();
        for (int blk = first; blk < wr.end; blk += NW) {
            const int k0 = blk * 32;
            f32x16 s = native_rowwise<D>(kptr + (int64_t)k0 * p.sk.t, p.sk.t, seq_len - k0, qptr + (int64_t)qb * p.sq.t, p.sq.t, seq_len - qb, lane);
            softmax(s, blk);
            native_transposed<D>(vptr + (int64_t)k0 * p.sv.t, p.sv.t, seq_len - k0, s, o, lane);
        }
        const float l_row = sum_across_halves(l_run);
        if (again) fwd_small_leave<DB>(mine, WAVE_BYTES, lane, o, m_run, l_row);
    }
    __syncthreads();
    fwd_small_merge<f32_t, D, NW>(p, smem, WAVE_BYTES, wave, lane, obase, lse_base, q_pos, seq_len);
}

}  // namespace chill
