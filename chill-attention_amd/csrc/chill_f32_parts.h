// fp32 matrix products on the bf16 matrix instructions, without a scale.
//
// An fp32 value is the sum of three bf16 values, high = bf16(x), mid = bf16(x - high), low = x - high - mid, each rounded to
// nearest: 3 x 8 bits hold the 24 of x, and bf16 has the exponent range of fp32, so the sum is exact down to 2^-109.  Of the nine
// products of two such sums the three smallest, mid low, low mid and low low, together less than 2^-24 of the whole (2 x 2^-8 x 2^-17
// and 2^-34), are left out.  v_mfma_f32_32x32x16_bf16 takes 32 cycles for 16 contraction
// steps, v_mfma_f32_32x32x2_f32 64 cycles for 2: the six products take 192 cycles where the fp32 instruction takes 512.  The
// split of an operand's eight values takes 44 vector instructions, which a wave issues between the MFMAs (SplitJob).  Every value
// has its own exponent: no scale is shared by a slice of rows, so what a row sees decides it and nothing else.
//
// An infinity has the parts inf and NaN, and so has a value that bf16(x) rounds beyond its range: sums that see one are NaN.  A
// wave that has such sums computes its blocks again with the fp32 instruction (native_rowwise, native_transposed), and the rows that
// have them take their result from there; the other rows keep theirs.
//
// Below 2^-109 the low part loses what lies under 2^-133, the smallest bf16.  P and dS, which come there by themselves, are scaled
// by 2^16 before their split, which then is exact for every fp32 value, and the sums over them by 2^-16 at the end.  Rows of
// Q, K, V and dO with bits below 2^-133 are noticed as they are split (SplitJob) and left to the fp32 instruction: by the waves whose
// blocks have them, or, where the row is a wave's own, for that row alone.  Forward / dQ / dK/dV in us without both -> with them, causal
// B4 H16 T4096 D64 720 / 940 / 1428 -> 720 / 942 / 1477, D32 389 / 521 / 712 -> 398 / 522 / 722, D128 1524 / 2084 / 2706 -> 1549 /
// 2014 / 2727, prefix-LM B1 H8 T2048 D64 53.4 / 61.8 / 81.8 -> 53.4 / 59.7 / 84.6.
#pragma once

#include "chill_device.h"
#include "chill_mask.h"
#include "chill_tiles.h"

namespace chill {

// One operand of v_mfma_f32_32x32x16_bf16 in its three parts.
struct Parts {
    i32x4 h, m, l;
};

// P and dS are split scaled by this (above)
constexpr float kPartsUp = 65536.f, kPartsDown = 1.f / 65536.f;

// The split of eight values, in the six shares that go behind the six MFMAs of the operand before: 44 instructions, in the order
// of the steps and not of the values, so that four others lie between an instruction and the one that needs its result (a wave
// on its own issues independent vector instructions every 5.3 cycles, dependent ones every 8).
// v_dot2_f32_bf16 with (-1, 0) and (0, -1) takes two of them in one, exactly, and is slower all the same (prefix-LM B1 H8 T2048
// D64, forward / dQ / dK/dV 61 / 71 / 90 -> 63 / 75 / 99 us): it waits for the MFMAs it stands between.
struct SplitJob {
    f32x8 x;
    Parts p;
    float up[8];  // the parts packed last, as floats
    template <int K>
    __device__ __forceinline__ void step() {
        constexpr int round = K / 20, k = K % 20;  // high parts, mid parts (20 instructions each), low parts
        i32x4& packed = round == 0 ? p.h : round == 1 ? p.m : p.l;
        if constexpr (k < 4) {
            packed[k] = Elem<bf16_t>::pack2(x[2 * k], x[2 * k + 1]);
        } else if constexpr (k < 12) {
            constexpr int i = k - 4;
            up[i] = __builtin_bit_cast(float, i % 2 == 0 ? packed[i / 2] << 16 : packed[i / 2] & 0xffff0000);
        } else {
            x[k - 12] -= up[k - 12];
        }
    }
    template <int SHARE>
    __device__ __forceinline__ void share() {
        constexpr int first = SHARE * 44 / 6, last = (SHARE + 1) * 44 / 6;
        static_for<last - first>([&](auto i) { step<first + i>(); });
    }
    __device__ __forceinline__ void all() {
        static_for<44>([&](auto i) { step<i>(); });
    }
    // The same with a look at what the low parts round (four instructions): bits of `lost` below the 16th say that one of them is no
    // bf16, which has the high 16.
    template <int SHARE>
    __device__ __forceinline__ void share(int& lost) {
        static_for<8>([&](auto i) { watched_step<8 * SHARE + i>(lost); });
    }
    __device__ __forceinline__ void all(int& lost) {
        static_for<48>([&](auto i) { watched_step<i>(lost); });
    }
    template <int K>
    __device__ __forceinline__ void watched_step(int& lost) {
        if constexpr (K < 44)
            step<K>();
        else
            lost |= __builtin_bit_cast(int, x[2 * (K - 44)]) | __builtin_bit_cast(int, x[2 * (K - 44) + 1]);
        // (here and not behind all splits, where what they round would have to be kept: dQ at head dim 128 spilled 73 registers)
        if constexpr (K == 47) asm volatile("" : "+v"(lost));
    }
    // holds the split where it stands (the compiler moves one that is used behind a branch there)
    __device__ __forceinline__ void pin() { asm volatile("" : "+v"(p.h), "+v"(p.m), "+v"(p.l)); }
};

// product K of the six of c += A B, the small ones first
template <int K>
__device__ __forceinline__ f32x16 mma_part(const Parts& a, const Parts& b, f32x16 c) {
    const i32x4 x = K == 0 ? a.l : (K == 2 || K == 3) ? a.m : a.h;
    const i32x4 y = K == 1 ? b.l : (K == 2 || K == 4) ? b.m : b.h;
    return Elem<bf16_t>::mma(x, y, c);
}

// the same products in the same order with the operands exchanged: c is the transposed sum, bit by bit
template <int K>
__device__ __forceinline__ f32x16 mma_part_transposed(const Parts& a, const Parts& b, f32x16 c) {
    return mma_part<K == 0 ? 1 : K == 1 ? 0 : K == 3 ? 4 : K == 4 ? 3 : K>(a, b, c);
}

// f(0), ..., f(N - 1), each left where it stands: one MFMA, and the vector and memory instructions that go behind it
template <int N, typename F>
__device__ __forceinline__ void slots(F&& f) {
    static_for<N>([&](auto i) {
        f(i);
        __builtin_amdgcn_sched_barrier(0);
    });
}

// 32 rows of fp32 in registers, a lane's half of its row (n, h): of operand j, which is 16 columns, the columns 16 j + 8 h .. + 7
template <int D>
struct F32Rows {
    static constexpr int N = D / 16;  // operands
    f32x4 c[2 * N];
    // the lane's part of row row0 + n; rows at and beyond `rows` repeat the last one (what is computed from them is masked)
    __device__ __forceinline__ static const float* at(const float* tensor, int64_t stride, int row0, int rows, int lane) {
        return tensor + (int64_t)imin(row0 + (lane & 31), rows - 1) * stride + 8 * (lane >> 5);
    }
    template <int J>
    __device__ __forceinline__ void load(const float* row) {
        c[2 * J] = *reinterpret_cast<const f32x4*>(row + 16 * J);
        c[2 * J + 1] = *reinterpret_cast<const f32x4*>(row + 16 * J + 4);
    }
    __device__ __forceinline__ void load_all(const float* row) {
        static_for<N>([&](auto j) { load<j>(row); });
    }
    template <int J>
    __device__ __forceinline__ f32x8 operand() const {
        return __builtin_shufflevector(c[2 * J], c[2 * J + 1], 0, 1, 2, 3, 4, 5, 6, 7);
    }
};

// rows that stay, split once
template <int D>
struct F32Resident {
    static constexpr int N = D / 16;
    Parts p[N];
    __device__ __forceinline__ void split(const F32Rows<D>& rows, int& lost) {
        static_for<N>([&](auto j) {
            SplitJob job;
            job.x = rows.template operand<j>();
            job.all(lost);
            p[j] = job.p;
        });
    }
    // (exact: see kPartsUp)
    __device__ __forceinline__ void split_scaled_up(const F32Rows<D>& rows) {
        static_for<N>([&](auto j) {
            SplitJob job;
            job.x = rows.template operand<j>() * kPartsUp;
            job.all();
            p[j] = job.p;
        });
    }
};

// the lanes whose splits have lost a bit
__device__ __forceinline__ uint64_t lanes_that_lost(int lost) { return __builtin_amdgcn_ballot_w64((lost & 0xffff) != 0); }
// whether row n, lanes n and n + 32, is among them
__device__ __forceinline__ bool row_that_lost(uint64_t lanes, int lane) {
    return (((uint32_t)lanes | (uint32_t)(lanes >> 32)) >> (lane & 31) & 1) != 0;
}

// The parts of 32 rows in LDS as three swizzled bf16 tiles, written row by row and read transposed.
template <int D>
struct F32Planes {
    typedef LdsTile<bf16_t, D> L;
    static constexpr int PLANE = L::bytes(32);
    static constexpr int BYTES = 3 * PLANE;
    // operand J of the lane's row: a share of three
    template <int J, int PART>
    __device__ __forceinline__ static void write(char* planes, const Parts& p, int lane) {
        *reinterpret_cast<i32x4*>(planes + PART * PLANE + L::chunk_off(lane & 31, 2 * J + (lane >> 5))) =
            PART == 0 ? p.h : PART == 1 ? p.m : p.l;
    }
    // the transposed operand of accumulator registers 8 s .. 8 s + 7 and head-dim block db
    __device__ __forceinline__ static Parts transposed(const lds_char* planes, const OperandOffsets<bf16_t, D>& ofs, int s, int db, int lane) {
        Parts p;
        p.h = ofs.tr_operand(planes, 0, s, db, lane);
        p.m = ofs.tr_operand(planes + PLANE, 0, s, db, lane);
        p.l = ofs.tr_operand(planes + 2 * PLANE, 0, s, db, lane);
        return p;
    }
};

// accumulator registers 8 s .. 8 s + 7: the values of a B operand
template <int S>
__device__ __forceinline__ f32x8 half_of(const f32x16& x) {
    return __builtin_shufflevector(x, x, 8 * S, 8 * S + 1, 8 * S + 2, 8 * S + 3, 8 * S + 4, 8 * S + 5, 8 * S + 6, 8 * S + 7);
}

// The mask of a block that is not predicate-free: entries no pair sees become `fill`.  `pos` = the lane's own row or key.
template <int MASK, bool QROWS>
__device__ __forceinline__ void mask_f32_block(f32x16& s, const Range& vis, int pos, int other0, int seq_len, MaskArgs a, int h, float fill) {
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

// P of a score: rounded after the scale as the forward does before it takes the largest as its reference, so that P of a row's
// largest comes out of it as it went into LSE2 (fused, dV of scores up to 50 was off by 1.06 times what the fp32 instruction left)
__device__ __forceinline__ float f32_probability(float s, float scale, float lse) {
#pragma clang fp contract(off)
    const float x = s * scale;
    return fast_exp2(x - lse);
}

// NaN in the lanes of a row (n, 0), (n, 1) that has an accumulator that is infinite or NaN, 0 in the others
template <int N>
__device__ __forceinline__ float nan_if_not_finite(const f32x16 (&acc)[N], float more = 0.f) {
    float t = more * 0.f;
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) t = __builtin_fmaf(acc[i][r], 0.f, t);
    return sum_across_halves(t);
}

template <int N>
__device__ __forceinline__ void scale_f32_blocks(f32x16 (&acc)[N], float by) {
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] *= by;
}

// ---------------------------------------------------------------- the fp32 instruction, operands from global memory
// X (32 rows) B^T (32 rows), both row-wise; rows behind x_rows and b_rows read as zero
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
// acc += X^T P, X 32 rows, P an accumulator block
template <int D>
__device__ __forceinline__ void native_transposed(const float* x, int64_t x_stride, int x_rows, const f32x16& p,
                                                  f32x16 (&acc)[(D + 31) / 32], int lane) {
    constexpr int DB = (D + 31) / 32;
    const int n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = 8 * (r / 4) + 4 * h + (r % 4);
#pragma unroll
        for (int db = 0; db < DB; db++) {
            const int col = D < 32 ? (n & (D - 1)) : 32 * db + n;
            const float a = row < x_rows ? x[(int64_t)row * x_stride + col] : 0.f;
            acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, p[r], acc[db], 0, 0, 0);
        }
    }
}

}  // namespace chill
