// dQ and dK/dV of fp32 launches with few 32-row tiles: as chill_f32_fwd_small.h does it for the forward.
#pragma once

#include "chill_bwd_small.h"
#include "chill_f32_parts.h"

namespace chill {

// ------------------------------------------------------------------------------------------ dQ
// (TILES as in dq_small_kernel)
template <int D, int MASK, int TILES>
__global__ __launch_bounds__(kFwdSmallWaves * 64 * TILES) __attribute__((amdgpu_waves_per_eu(TILES))) void dq_small_f32_kernel(BwdParams p, int n_q_tiles, int total_items, int has_full_blocks) {
    constexpr int NW = kFwdSmallWaves, NT = NW * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int WAVE_BYTES = bwd_small_wave_bytes(D, CHILL_F32, 1, true);
    extern __shared__ __attribute__((aligned(16))) char smem_all[];
    const int item = blockIdx.x;
    if (item >= total_items) return;
    const int half = TILES == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;  // which block of the workgroup
    char* smem = smem_all + half * (NW * WAVE_BYTES);
    // the blocks of all heads from the long end to the short end (under causal-like masks: longest first)
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
    float* dqbase = reinterpret_cast<float*>(p.dq) + b * p.sdq.b + hd * p.sdq.h;
    if (!has_tile || qb >= seq_len) {
        if (has_tile) {
            // rows at or beyond lens[b] receive 0 (the reference relies on the adapter's zero-fill, chill.py:292)
            const int nrows = imin(32, p.T - qb);
            zero_rows<f32_t, D, NT>(dqbase, p.sdq.t, qb, nrows, tid);
            // (the dK/dV launch that follows reads delta of every row of the tiles it visits)
            if (p.delta_out != nullptr)
                for (int i = tid; i < nrows; i += NT) p.delta_out[b * p.delta_b + hd * p.delta_h + qb + i] = 0.f;
        }
        if constexpr (TILES == 2) __syncthreads();  // the other half's one barrier
        return;
    }
    const float* qptr = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hd * p.sq.h;
    const float* doptr = reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hd * p.sdo.h;
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h;

    // the 32-key blocks of these rows (utils.py:221-272 with 32 x 32 tiles)
    const TileRange wr = tile_range<MASK, true>(qb, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    const int first = wr.start + wave;
    const int q_pos = qb + n;
    F32Rows<D> kv;  // K of the block that is due, then its V, then the next block's K
    F32Resident<D> q, d_o;
    float lse_q = 0.f, delta_q = 0.f;
    int lost = 0;  // (of K and V)
    uint64_t lost_rows;
    {
        F32Rows<D> rows;
        rows.load_all(F32Rows<D>::at(doptr, p.sdo.t, qb, seq_len, lane));
        if (q_pos < p.T) lse_q = p.lse[b * p.lse_b + hd * p.lse_h + q_pos];
        if (p.delta_out != nullptr) {
            // delta = rowsum(O * dO), 0 for rows past the sequence (the rows here repeat the last one); every wave of the workgroup
            // holds the same 32 rows, the first one writes
            F32Rows<D> out;
            const float* optr = reinterpret_cast<const float*>(p.o) + b * p.so.b + hd * p.so.h;
            out.load_all(F32Rows<D>::at(optr, p.so.t, qb, seq_len, lane));
#pragma unroll
            for (int i = 0; i < 2 * N; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) delta_q += out.c[i][e] * rows.c[i][e];
            delta_q += __shfl_xor(delta_q, 32, 64);
            if (q_pos >= seq_len) delta_q = 0.f;
            if (wave == 0 && h == 0 && q_pos < p.T) p.delta_out[b * p.delta_b + hd * p.delta_h + q_pos] = delta_q;
        } else if (q_pos < p.T) {
            delta_q = p.delta[b * p.delta_b + hd * p.delta_h + q_pos];
        }
        d_o.split_scaled_up(rows);
        rows.load_all(F32Rows<D>::at(qptr, p.sq.t, qb, seq_len, lane));
        const int blk = imax(imin(first, wr.end - 1), 0);  // (a wave without blocks loads one all the same)
        kv.load_all(F32Rows<D>::at(kptr, p.sk.t, blk * 32, seq_len, lane));
        int lost_q = 0;
        q.split(rows, lost_q);
        lost_rows = lanes_that_lost(lost_q);
    }
    // a row that attends to nothing has LSE2 = -inf and only masked entries (score -inf): P = exp2(-inf - 0)
    if (lse_q == -INFINITY) lse_q = 0.f;
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);
    char* mine = smem + wave * WAVE_BYTES;
    const lds_char* planes = (const lds_char*)mine;
    // Two waves a SIMD have 256 registers each, 12 too few at head dim 64.  The low parts of dO lie in LDS, behind the planes: a register reloaded
    // from scratch memory waits for every row of K and V requested before it (prefix-LM B1 H8 T2048
    // 71.6 -> 67.7 us, causal B1 H2 T8192 217 -> 167; one is left)
    constexpr bool kParked = TILES == 2 && D == 64;
    constexpr int PARKED = 64 * 16;
    static_assert(!kParked || Planes::BYTES + N * PARKED <= WAVE_BYTES, "room behind the planes");
    if constexpr (kParked)
        static_for<N>([&](auto j) { *reinterpret_cast<i32x4*>(mine + Planes::BYTES + j * PARKED + lane * 16) = d_o.p[j].l; });

    f32x16 dq[DB];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < DB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) dq[i][r] = 0.f;
    };
    clear();
    const Range vis = visible_range<MASK, true>(q_pos, seq_len, p.margs);
    const float scale = p.scale_log2;
    const float masked_score = scale < 0.f ? INFINITY : -INFINITY;  // times the scale: -inf
    auto mask = [&](f32x16& s, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, true>(s, vis, q_pos, blk * 32, seq_len, p.margs, h, masked_score);
    };

    SplitJob job[2];
    job[0].x = kv.template operand<0>();
    job[0].all(lost);
    for (int blk = first; blk < wr.end; blk += NW) {
        const int next = blk + NW < wr.end ? blk + NW : blk;
        const float* k_next = F32Rows<D>::at(kptr, p.sk.t, next * 32, seq_len, lane);
        const float* v_row = F32Rows<D>::at(vptr, p.sv.t, blk * 32, seq_len, lane);
        f32x16 s, dp;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = 0.f;
            dp[r] = -delta_q * kPartsUp;
        }
        // S^T and, scaled up, dP^T blocks: rows = keys 8 * (r / 4) + 4 * h + r % 4 of the block, column n = query row.  Operand t, K's and
        // then V's, in job[t % 2]; its successor is split behind its MFMAs
        i32x4 low;
        auto operand_slot = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value, t = i / 6, part = i % 6;
            if constexpr (t < N)
                s = mma_part<part>(job[t % 2].p, q.p[t % N], s);
            else if constexpr (kParked)
                dp = mma_part<part>(job[t % 2].p, Parts{d_o.p[t % N].h, d_o.p[t % N].m, low}, dp);
            else
                dp = mma_part<part>(job[t % 2].p, d_o.p[t % N], dp);
            constexpr int u = t + 1;
            if constexpr (kParked && part == 2 && u >= N && u < 2 * N)
                low = *reinterpret_cast<const lds_i32x4*>(planes + Planes::BYTES + (u - N) * PARKED + lane * 16);
            if constexpr (t == 0 && part == 0) kv.template load<0>(v_row);
            if constexpr (u < 2 * N) {
                if constexpr (part == 0) job[u % 2].x = kv.template operand<u % N>();
                job[u % 2].template share<part>(lost);
                if constexpr (part == 5 && u == N) job[u % 2].pin();
                // (what is due a phase later takes the place of the rows just split)
                if constexpr (part == 2) kv.template load<u % N>(u < N ? v_row : k_next);
            }
            if constexpr (t < N && part < 3) Planes::template write<t % N, part>(mine, job[t % 2].p, lane);
        };
        slots<6 * N>([&](auto i) { operand_slot(i); });
        mask(s, blk);
        constexpr int PER = (16 + 6 * N - 1) / (6 * N);  // exponentials a slot
        Parts kt[2];
        slots<6 * N>([&](auto i) {
            operand_slot(std::integral_constant<int, 6 * N + i>{});
#pragma unroll
            for (int r = PER * i; r < PER * (i + 1) && r < 16; r++) s[r] = f32_probability(s[r], scale, lse_q);
            if constexpr (i == 6 * N - 3) kt[0] = Planes::transposed(planes, ofs, 0, 0, lane);
        });
#pragma unroll
        for (int r = 0; r < 16; r++) dp[r] *= s[r];
        job[0].x = half_of<0>(dp);
        job[0].all();
        job[1].x = half_of<1>(dp);
        __builtin_amdgcn_sched_barrier(0);
        // dQ^T += K^T dS^T: the halves of dS in job[0] and job[1], the second one split beside the first one's MFMAs, the first
        // operand of the next block beside the second one's
        slots<12 * DB>([&](auto i) {
            constexpr int step = i / 6, part = i % 6, half = step / DB, db = step % DB;
            dq[db] = mma_part<part>(kt[step % 2], job[half].p, dq[db]);
            if constexpr (part == 0 && step + 1 < 2 * DB)
                kt[(step + 1) % 2] = Planes::transposed(planes, ofs, (step + 1) / DB, (step + 1) % DB, lane);
            if constexpr (step == 0) job[1].template share<part>();
            if constexpr (step == DB) {
                if constexpr (part == 0) job[0].x = kv.template operand<0>();
                job[0].template share<part>(lost);
            }
        });
    }
    scale_f32_blocks(dq, kPartsDown);
    bwd_small_leave<DB>(mine, 0, dq, lane);
    const float bad = nan_if_not_finite(dq);
    const bool again = bad != bad || row_that_lost(lost_rows, lane) || lanes_that_lost(lost) != 0;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear();
        for (int blk = first; blk < wr.end; blk += NW) {
            const int k0 = blk * 32;
            const float *kb = kptr + (int64_t)k0 * p.sk.t, *vb = vptr + (int64_t)k0 * p.sv.t;
            f32x16 s = native_rowwise<D>(kb, p.sk.t, seq_len - k0, qptr + (int64_t)qb * p.sq.t, p.sq.t, seq_len - qb, lane);
            f32x16 dp = native_rowwise<D>(vb, p.sv.t, seq_len - k0, doptr + (int64_t)qb * p.sdo.t, p.sdo.t, seq_len - qb, lane);
            mask(s, blk);
#pragma unroll
            for (int r = 0; r < 16; r++) dp[r] = f32_probability(s[r], scale, lse_q) * (dp[r] - delta_q);
            native_transposed<D>(kb, p.sk.t, seq_len - k0, dp, dq, lane);
        }
        if (again) bwd_small_leave<DB>(mine, 0, dq, lane);
    }
    __syncthreads();
    float* const rows[1] = {dqbase + (int64_t)q_pos * p.sdq.t};
    const float mult[1] = {p.sm_scale};
    bwd_small_merge<f32_t, D, 1, NW>(smem, WAVE_BYTES, wave, lane, rows, mult, q_pos < p.T, q_pos < seq_len);
}

// ------------------------------------------------------------------------------------------ dK, dV
template <int D, int MASK>
__global__ __launch_bounds__(kFwdSmallWaves * 64) void dkdv_small_f32_kernel(BwdParams p, int n_k_tiles, int total_items, int has_full_blocks) {
    constexpr int NW = kFwdSmallWaves, NT = NW * 64, DB = (D + 31) / 32, N = D / 16;
    typedef F32Planes<D> Planes;
    constexpr int WAVE_BYTES = bwd_small_wave_bytes(D, CHILL_F32, 2, true);
    constexpr int VEC_OFF = WAVE_BYTES - 2 * 32 * 4;  // LSE2 and -delta of a block's query rows
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int item = blockIdx.x;
    if (item >= total_items) return;
    // the key blocks of all heads from the first to the last (under causal-like masks: longest first)
    const int n_heads = total_items / n_k_tiles;
    const int bh = item % n_heads, kt_index = item / n_heads;
    const int b = bh / p.H_kv, hkv = bh % p.H_kv;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    int seq_len = p.T;
    if (p.lens != nullptr) seq_len = imin(p.lens[(int64_t)b * p.lens_stride], p.T);

    const int kb0 = kt_index * 32;
    float* dkbase = reinterpret_cast<float*>(p.dk) + b * p.sdk.b + hkv * p.sdk.h;
    float* dvbase = reinterpret_cast<float*>(p.dv) + b * p.sdv.b + hkv * p.sdv.h;
    if (kb0 >= seq_len) {
        // rows at or beyond lens[b] receive 0 (the reference relies on the adapter's zero-fill, chill.py:293-294)
        const int nrows = imin(32, p.T - kb0);
        zero_rows<f32_t, D, NT>(dkbase, p.sdk.t, kb0, nrows, tid);
        zero_rows<f32_t, D, NT>(dvbase, p.sdv.t, kb0, nrows, tid);
        return;
    }
    // the 32-query blocks that see these keys
    const TileRange wr = tile_range<MASK, false>(kb0, 32, 32, seq_len, has_full_blocks != 0, p.margs);
    const int n_blocks = wr.end - wr.start;
    const int n_iters = n_blocks * p.group;  // every query head of the GQA group in turn (chill_bwd_dkdv.py:156)

    // iteration it = (group head, query block)
    auto q_rows = [&](int it) {
        const int hq = hkv * p.group + it / n_blocks;
        return F32Rows<D>::at(reinterpret_cast<const float*>(p.q) + b * p.sq.b + hq * p.sq.h, p.sq.t, (wr.start + it % n_blocks) * 32, seq_len, lane);
    };
    auto do_rows = [&](int it) {
        const int hq = hkv * p.group + it / n_blocks;
        return F32Rows<D>::at(reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hq * p.sdo.h, p.sdo.t, (wr.start + it % n_blocks) * 32, seq_len, lane);
    };
    // LSE2 (lanes 0..31) and delta (lanes 32..63) of the block's rows; rows past the sequence repeat the last one, as those of Q and dO
    // do (no key sees them)
    auto row_vec = [&](int it) {
        const int hq = hkv * p.group + it / n_blocks, q = (wr.start + it % n_blocks) * 32 + n;
        const float* src = h == 0 ? p.lse + b * p.lse_b + hq * p.lse_h : p.delta + b * p.delta_b + hq * p.delta_h;
        return src[imin(q, seq_len - 1)];
    };
    const float* kptr = reinterpret_cast<const float*>(p.k) + b * p.sk.b + hkv * p.sk.h + (int64_t)kb0 * p.sk.t;
    const float* vptr = reinterpret_cast<const float*>(p.v) + b * p.sv.b + hkv * p.sv.h + (int64_t)kb0 * p.sv.t;
    F32Rows<D> q, d_o;
    F32Resident<D> k, v;
    float vec_next = 0.f;
    int lost = 0;  // (of Q and dO)
    uint64_t lost_rows;
    {
        F32Rows<D> kr, vr;
        kr.load_all(F32Rows<D>::at(kptr, p.sk.t, 0, seq_len - kb0, lane));
        vr.load_all(F32Rows<D>::at(vptr, p.sv.t, 0, seq_len - kb0, lane));
        if (wave < n_iters) {
            q.load_all(q_rows(wave));
            d_o.load_all(do_rows(wave));
            vec_next = row_vec(wave);
        }
        int lost_kv = 0;
        k.split(kr, lost_kv);
        v.split(vr, lost_kv);
        lost_rows = lanes_that_lost(lost_kv);
    }
    const int k_pos = kb0 + n;
    const Range vis = visible_range<MASK, false>(k_pos, seq_len, p.margs);
    OperandOffsets<bf16_t, D> ofs;
    ofs.init(lane);
    char* mine = smem + wave * WAVE_BYTES;
    const lds_char *q_planes = (const lds_char*)mine, *do_planes = q_planes + Planes::BYTES;
    const lds_float* vec = reinterpret_cast<const lds_float*>((const lds_char*)mine + VEC_OFF);

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
    const float scale = p.scale_log2;
    const float masked_score = scale < 0.f ? INFINITY : -INFINITY;  // times the scale: -inf
    auto mask = [&](f32x16& s, int blk) {
        if (!(blk >= wr.full_start && blk < wr.full_end))
            mask_f32_block<MASK, false>(s, vis, k_pos, blk * 32, seq_len, p.margs, h, masked_score);
    };
    // LSE2 and -delta of the rows of this lane's accumulator registers, through LDS
    auto leave_vec = [&](float x) {
        // (a row that attends to nothing has LSE2 = -inf and only masked entries)
        reinterpret_cast<float*>(mine + VEC_OFF)[lane] = h == 0 ? (x == -INFINITY ? 0.f : x) : -x;
    };
    auto read_vec = [&](int at) {
        f32x16 x;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const f32x4 y = *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(vec + at + 8 * g + 4 * h);
#pragma unroll
            for (int e = 0; e < 4; e++) x[4 * g + e] = y[e];
        }
        return x;
    };

    SplitJob job[2];
    if (wave < n_iters) {
        job[0].x = q.template operand<0>();
        job[0].all(lost);
    }
    for (int it = wave; it < n_iters; it += NW) {
        const int blk = wr.start + it % n_blocks;
        const int next = it + NW < n_iters ? it + NW : it;
        const float *q_next = q_rows(next), *do_next = do_rows(next);
        leave_vec(vec_next);
        vec_next = row_vec(next);
        f32x16 s, dp = read_vec(32);  // (the dP chain starts from -delta)
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.f;
        // S (rounded as in the forward) and dP blocks: rows = queries 8 * (r / 4) + 4 * h + r % 4 of the block, column n = key.  Operand t, Q's and then
        // dO's, in job[t % 2]; its successor is split behind its MFMAs
        auto operand_slot = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value, t = i / 6, part = i % 6;
            if constexpr (t < N)
                s = mma_part_transposed<part>(job[t % 2].p, k.p[t % N], s);
            else
                dp = mma_part<part>(job[t % 2].p, v.p[t % N], dp);
            constexpr int u = t + 1;
            if constexpr (u < 2 * N) {
                if constexpr (part == 0) {
                    if constexpr (u < N)
                        job[u % 2].x = q.template operand<u % N>();
                    else
                        job[u % 2].x = d_o.template operand<u % N>();
                }
                job[u % 2].template share<part>(lost);
                if constexpr (part == 5 && u == N) job[u % 2].pin();
                // (the rows of the next block take the place of those just split)
                if constexpr (part == 2 && u < N) q.template load<u % N>(q_next);
                if constexpr (part == 2 && u >= N) d_o.template load<u % N>(do_next);
            }
            if constexpr (t == 0 && part == 0) q.template load<0>(q_next);
            if constexpr (part < 3) Planes::template write<t % N, part>(mine + (t < N ? 0 : Planes::BYTES), job[t % 2].p, lane);
        };
        slots<6 * N>([&](auto i) { operand_slot(i); });
        const f32x16 lse = read_vec(0);
        mask(s, blk);
        // the exponentials (P, and with it dS, scaled up) of the first half of P in the first half of the dP chain, so that it can be split in the last step
        SplitJob pj[2];
        constexpr int PER = (16 + 6 * N - 7) / (6 * N - 6 > 0 ? 6 * N - 6 : 1);
        slots<6 * N>([&](auto i) {
            operand_slot(std::integral_constant<int, 6 * N + i>{});
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
        Parts tr[2];
        tr[0] = Planes::transposed(do_planes, ofs, 0, 0, lane);
        __builtin_amdgcn_sched_barrier(0);
        // dV^T += dO^T P, then dK^T += Q^T dS; step w of 4 DB.  Beside them: the second half of P, dS and its two halves, and the
        // first operand of the next block
        slots<24 * DB>([&](auto i) {
            constexpr int w = i / 6, part = i % 6, half = w / DB % 2, db = w % DB;
            if constexpr (w < 2 * DB)
                dv[db] = mma_part<part>(tr[w % 2], pj[half].p, dv[db]);
            else
                dk[db] = mma_part<part>(tr[w % 2], pj[half].p, dk[db]);
            if constexpr (part == 0 && w + 1 < 4 * DB)
                tr[(w + 1) % 2] = Planes::transposed(w + 1 < 2 * DB ? do_planes : q_planes, ofs, (w + 1) / DB % 2, (w + 1) % DB, lane);
            if constexpr (w == 0) {
                pj[1].template share<part>();
#pragma unroll
                for (int r = 3 * part; r < 3 * part + 3 && r < 16; r++) dp[r] *= s[r];
            }
            // (pj[0] is free behind the first half of dV's MFMAs, pj[1] behind the second)
            if constexpr (w == DB) {
                if constexpr (part == 0) pj[0].x = half_of<0>(dp);
                pj[0].template share<part>();
            }
            if constexpr (w == 2 * DB) {
                if constexpr (part == 0) pj[1].x = half_of<1>(dp);
                pj[1].template share<part>();
            }
            if constexpr (w == 3 * DB) {
                if constexpr (part == 0) job[0].x = q.template operand<0>();
                job[0].template share<part>(lost);
            }
        });
    }
    scale_f32_blocks(dk, kPartsDown);
    scale_f32_blocks(dv, kPartsDown);
    bwd_small_leave<DB>(mine, 0, dk, lane);
    bwd_small_leave<DB>(mine, DB, dv, lane);
    const float bad = nan_if_not_finite(dk, nan_if_not_finite(dv));
    const bool again = bad != bad || row_that_lost(lost_rows, lane) || lanes_that_lost(lost) != 0;
    if (__builtin_amdgcn_ballot_w64(again) != 0) {
        clear();
        for (int it = wave; it < n_iters; it += NW) {
            const int hq = hkv * p.group + it / n_blocks, blk = wr.start + it % n_blocks, q0 = blk * 32;
            const float* qb = reinterpret_cast<const float*>(p.q) + b * p.sq.b + hq * p.sq.h + (int64_t)q0 * p.sq.t;
            const float* dob = reinterpret_cast<const float*>(p.d_o) + b * p.sdo.b + hq * p.sdo.h + (int64_t)q0 * p.sdo.t;
            leave_vec(row_vec(it));
            f32x16 s = native_rowwise<D>(qb, p.sq.t, seq_len - q0, kptr, p.sk.t, seq_len - kb0, lane);
            f32x16 dp = native_rowwise<D>(dob, p.sdo.t, seq_len - q0, vptr, p.sv.t, seq_len - kb0, lane);
            const f32x16 lse = read_vec(0), neg_delta = read_vec(32);
            mask(s, blk);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                s[r] = f32_probability(s[r], scale, lse[r]);
                dp[r] = s[r] * (dp[r] + neg_delta[r]);
            }
            native_transposed<D>(dob, p.sdo.t, seq_len - q0, s, dv, lane);
            native_transposed<D>(qb, p.sq.t, seq_len - q0, dp, dk, lane);
        }
        if (again) {
            bwd_small_leave<DB>(mine, 0, dk, lane);
            bwd_small_leave<DB>(mine, DB, dv, lane);
        }
    }
    __syncthreads();
    float* const rows[2] = {dkbase + (int64_t)k_pos * p.sdk.t, dvbase + (int64_t)k_pos * p.sdv.t};
    const float mult[2] = {p.sm_scale, 1.f};
    bwd_small_merge<f32_t, D, 2, NW>(smem, WAVE_BYTES, wave, lane, rows, mult, k_pos < p.T, k_pos < seq_len);
}

}  // namespace chill
