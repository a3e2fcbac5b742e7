// fp32 matrix products on the fp16 matrix instructions.
//
// A block of fp32 values is scaled by a power of two that takes its largest magnitude to [2^14, 2^15), and each scaled value is
// held as the sum of two fp16 values, hi = fp16(x) and lo = fp16(x - hi): 22 significant bits and a sign, an error of at most
// 2^-23 of the value, or 2^-40 of the block's largest for values below 2^-17 of that.  Of the four products of two such
// sums lo * lo, at most 2^-22 and on average 2^-27 of the whole, is left out.  v_mfma_f32_32x32x16_f16 takes 32 cycles for 16
// contraction steps, v_mfma_f32_32x32x2_f32 64 cycles for 2: the three products take 96 cycles where the fp32 instruction
// takes 512.  They accumulate in fp32, in fewer roundings than the fp32 instruction makes: relative errors against 64 bits (2-norm;
// causal, T4096 D64) are 3.2e-7 / 3.9e-7 / 7.4e-7 / 7.3e-7 for O, dQ, dK, dV where the fp32 instruction gives 5.0e-7 / 5.0e-7 /
// 1.1e-6 / 1.1e-6, and no larger than its in any of 40 shapes (five masks, head dims 32 to 128, T 256 .. 4096).
// Infinities and NaN come out as NaN: callers check their finished sums and repeat what is not finite with the fp32
// instruction.
//
// A scale is kept as the exponent field of its fp32 representation (at most kPartsHigh; a larger field belongs to smaller
// values), so that scales multiply and divide by adding and subtracting fields.
#pragma once

#include "chill_device.h"

namespace chill {

constexpr int kPartsHigh = 253;  // (254 - field, the inverse, must be a normal number too)

// 2^(field - 127), 0 for fields below the normal range
__device__ __forceinline__ float pow2_of_field(int field) { return __builtin_bit_cast(float, (field < 0 ? 0 : field) << 23); }
// the scale of a block whose largest magnitude is x (given as its bits)
__device__ __forceinline__ int parts_field(int max_bits) {
    const int field = 127 + 14 + 127 - (int)((unsigned)max_bits >> 23);
    return field < kPartsHigh ? field : kPartsHigh;
}
__device__ __forceinline__ float parts_inverse(int field) { return __builtin_bit_cast(float, (254 - field) << 23); }

// max of |x| over the lanes, from the bits of every lane's non-negative maximum
__device__ __forceinline__ int max_across_wave(int bits) {
    auto step = [&](auto control) {
        const int other = __builtin_amdgcn_update_dpp(0, bits, decltype(control)::value, 0xf, 0xf, true);
        bits = other > bits ? other : bits;
    };
    step(std::integral_constant<int, 0xb1>{});   // quad_perm [1, 0, 3, 2]
    step(std::integral_constant<int, 0x4e>{});   // quad_perm [2, 3, 0, 1]
    step(std::integral_constant<int, 0x141>{});  // row_half_mirror
    step(std::integral_constant<int, 0x140>{});  // row_mirror
    auto a = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
    bits = (int)a[0] > (int)a[1] ? (int)a[0] : (int)a[1];
    a = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    bits = (int)a[0] > (int)a[1] ? (int)a[0] : (int)a[1];
    return __builtin_amdgcn_readfirstlane(bits);
}
__device__ __forceinline__ int max_bits_across_halves(int bits) {
    const auto a = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
    return (int)a[0] > (int)a[1] ? (int)a[0] : (int)a[1];
}

// max(acc, |x|, |y|) of non-negative acc.  (In asm: the compiler's fmax quiets every operand first.  The wait states are those
// a following cross-lane instruction needs, which the compiler does not count behind an asm statement.)
__device__ __forceinline__ float max3_abs(float acc, float x, float y) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(acc) : "v"(x), "v"(y));
    return acc;
}
__device__ __forceinline__ int max_bits(float acc) {
    asm("s_nop 1" : "+v"(acc));
    return __builtin_bit_cast(int, acc);
}

// The parts of four values times a scale, packed in pairs, in the eight instructions it takes (the compiler computes one hi of
// a pair twice).  An instruction that reads a register of which the one before wrote the upper half needs a wait state between
// them, and an MFMA two behind any vector instruction that wrote its operand: `TAIL` adds those; without it the results must
// go to LDS.
#define CHILL_SPLIT_QUAD(TAIL, KIND)                                                                                             \
    asm("v_fma_mixlo_f16 %0, %4, %8, 0\n\t"                                                                                      \
        "v_fma_mixlo_f16 %1, %6, %8, 0\n\t"                                                                                      \
        "v_fma_mixhi_f16 %0, %5, %8, 0\n\t"                                                                                      \
        "v_fma_mixhi_f16 %1, %7, %8, 0\n\t"                                                                                      \
        "v_fma_mixlo_f16 %2, %4, %8, -%0 op_sel_hi:[0,0,1]\n\t"                                                                  \
        "v_fma_mixlo_f16 %3, %6, %8, -%1 op_sel_hi:[0,0,1]\n\t"                                                                  \
        "v_fma_mixhi_f16 %2, %5, %8, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"                                                   \
        "v_fma_mixhi_f16 %3, %7, %8, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]" TAIL                                                  \
        : "=&v"(h0), "=&v"(h1), "=&v"(l0), "=&v"(l1)                                                                             \
        : "v"(x0), "v"(x1), "v"(x2), "v"(x3), KIND(scale))
__device__ __forceinline__ void split_quad_for_lds(f32x4 x, float scale, i32x2& hi, i32x2& lo) {
    const float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
    int h0, h1, l0, l1;
    CHILL_SPLIT_QUAD("", "s");
    hi = i32x2{h0, h1};
    lo = i32x2{l0, l1};
}
__device__ __forceinline__ void split_quad(float x0, float x1, float x2, float x3, float scale, i32x2& hi, i32x2& lo) {
    int h0, h1, l0, l1;
    CHILL_SPLIT_QUAD("\n\ts_nop 1", "v");
    hi = i32x2{h0, h1};
    lo = i32x2{l0, l1};
}
#undef CHILL_SPLIT_QUAD

// One operand of v_mfma_f32_32x32x16_f16 in its two parts.
struct Parts {
    i32x4 hi, lo;
};

__device__ __forceinline__ Parts split8(const float (&x)[8], float scale) {
    i32x2 h0, l0, h1, l1;
    split_quad(x[0], x[1], x[2], x[3], scale, h0, l0);
    split_quad(x[4], x[5], x[6], x[7], scale, h1, l1);
    return Parts{{h0[0], h0[1], h1[0], h1[1]}, {l0[0], l0[1], l1[0], l1[1]}};
}

// c += A B
__device__ __forceinline__ f32x16 mma_parts(const Parts& a, const Parts& b, f32x16 c) {
    c = Elem<f16_t>::mma(a.lo, b.hi, c);
    c = Elem<f16_t>::mma(a.hi, b.lo, c);
    return Elem<f16_t>::mma(a.hi, b.hi, c);
}

// 32 rows of D floats in LDS as two swizzled fp16 tiles, the hi parts first: as many bytes as the floats take.
template <int D>
struct PartTile {
    typedef LdsTile<f16_t, D> L;
    static constexpr int PLANE = L::bytes(32);
    static constexpr int BYTES = 2 * PLANE;
};

// ROWS rows of a 32-row block on their way from global memory through a wave's registers to a PartTile.  `fetch` requests rows
// row0 .. of a sequence of T rows (rows past its end repeat the last one: the caller masks what it computes from them, and what
// a tensor holds behind a shorter sequence must not set the scale), `measure` finds their scale, `commit<I>` writes the parts of
// the I-th of STEPS shares to the tile.
template <int D, int ROWS>
struct PartStager {
    static constexpr int CH = D / 4;             // 16-byte chunks of an fp32 row
    static constexpr int STEP_ROWS = 64 / CH;    // rows one step of the wave covers
    static constexpr int STEPS = ROWS / STEP_ROWS;
    static_assert(64 % CH == 0 && ROWS % STEP_ROWS == 0, "whole steps");
    f32x4 regs[STEPS];
    int field = 0;  // of the scale

    __device__ __forceinline__ void fetch(const float* tensor, int64_t row_stride, int row0, int T, int lane) {
        const int first = imin(row0, T - 1), last = T - 1 - first;
        const char* base = reinterpret_cast<const char*>(tensor + first * row_stride);
        const int row = lane / CH, c = lane % CH;
        const unsigned stride = (unsigned)row_stride * 4u;  // (below 2^23: the launchers refuse more)
#pragma unroll
        for (int i = 0; i < STEPS; i++)
            regs[i] = *reinterpret_cast<const f32x4*>(base + (__umul24((unsigned)imin(row + i * STEP_ROWS, last), stride) + 16u * c));
    }
    __device__ __forceinline__ void measure() {
        float m0 = 0.f, m1 = 0.f;
#pragma unroll
        for (int i = 0; i < STEPS; i++) {
            m0 = max3_abs(m0, regs[i][0], regs[i][1]);
            m1 = max3_abs(m1, regs[i][2], regs[i][3]);
        }
        field = parts_field(max_across_wave(max_bits(max3_abs(m0, m1, m1))));
    }
    // `row0`: the first row's place in the tile
    template <int I>
    __device__ __forceinline__ void commit(char* tile, int row0, int lane) const {
        typedef PartTile<D> P;
        const float scale = uniform(pow2_of_field(field));
        i32x2 hi, lo;
        split_quad_for_lds(regs[I], scale, hi, lo);
        char* dst = tile + P::L::elem_off(row0 + I * STEP_ROWS + lane / CH, 4 * (lane % CH));
        *reinterpret_cast<i32x2*>(dst) = hi;
        *reinterpret_cast<i32x2*>(dst + P::PLANE) = lo;
    }
};

// The wave's 32 resident rows as B operands, every row with a scale of its own: step t of the contraction takes columns
// 16 t + 8 h .. + 7 of row n.
template <int D>
struct ResidentParts {
    Parts c[D / 16];
    float inverse;  // of the scale of the lane's row

    // (times `sign`, 1 or -1)
    __device__ __forceinline__ void load(const float* base, int64_t row_stride, int rows_valid, int lane, float sign = 1.f) {
        const int n = lane & 31, h = lane >> 5;
        f32x4 x[D / 8];
        float m = 0.f;
#pragma unroll
        for (int t = 0; t < D / 8; t++) {
            x[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (n < rows_valid)
                x[t] = *reinterpret_cast<const f32x4*>(base + (int64_t)n * row_stride + 16 * (t / 2) + 8 * h + 4 * (t % 2));
        }
#pragma unroll
        for (int t = 0; t < D / 8; t++) m = max3_abs(max3_abs(m, x[t][0], x[t][1]), x[t][2], x[t][3]);
        const int field = parts_field(max_bits_across_halves(max_bits(m)));
        const float scale = pow2_of_field(field) * sign;
        inverse = parts_inverse(field);
#pragma unroll
        for (int t = 0; t < D / 16; t++) {
            const f32x4 a = x[2 * t], b = x[2 * t + 1];
            const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
            c[t] = split8(v, scale);
        }
    }
};

// acc(32 rows of the tile x 32 cols) += X B^T, B = resident rows.  Operands are read two steps ahead of their MFMAs, in this
// order and no other (the compiler would read each one right before its MFMA and wait for it); `beside(t)` is issued among the
// MFMAs of step t.
constexpr int kPartsAhead = 2;
template <int D, typename Beside>
__device__ __forceinline__ f32x16 mma_rowwise_parts(const lds_char* tile, const OperandOffsets<f16_t, D>& ofs,
                                                    const ResidentParts<D>& b, f32x16 acc, int lane, Beside&& beside) {
    constexpr int N = D / 16;
    Parts a[N];
    auto read = [&](auto t) {
        if constexpr (t < N) a[t] = Parts{ofs.row_chunk(tile, 0, t, lane), ofs.row_chunk(tile + PartTile<D>::PLANE, 0, t, lane)};
    };
    static_for<kPartsAhead>([&](auto t) { read(t); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<N>([&](auto t) {
        acc = mma_parts(a[t], b.c[t], acc);
        asm volatile("" : "+v"(acc));  // keeps the MFMAs at this place
        read(std::integral_constant<int, t + kPartsAhead>{});
        beside(t);
        __builtin_amdgcn_sched_barrier(0);
    });
    return acc;
}

// acc(32 columns of the tile x 32 cols, for NB 32-wide head-dim blocks from db0 on) += X^T P, P a 32x32 accumulator block whose
// rows are scaled by slices of 32 / SLICES.  The operands of X are read ahead as well, the first ones by `begin`, before P is known.
template <int D, int READ_AHEAD, int NB = (D + 31) / 32>
struct TransposedParts {
    static constexpr int N = 2 * NB;  // step u: 16 rows u / NB, head-dim block u % NB
    static constexpr int AHEAD = N < READ_AHEAD ? N : READ_AHEAD;
    Parts a[N];
    const lds_char* tile;  // (of the first head-dim block)
    const OperandOffsets<f16_t, D>& ofs;
    int lane;
    template <int U>
    __device__ __forceinline__ void read() {
        if constexpr (U < N)
            a[U] = Parts{ofs.tr_operand(tile, 0, U / NB, U % NB, lane), ofs.tr_operand(tile + PartTile<D>::PLANE, 0, U / NB, U % NB, lane)};
    }
    __device__ __forceinline__ TransposedParts(const lds_char* t, const OperandOffsets<f16_t, D>& o, int l) : tile(t), ofs(o), lane(l) {}
    __device__ __forceinline__ void begin() {
        static_for<AHEAD>([&](auto u) { read<u>(); });
        __builtin_amdgcn_sched_barrier(0);
    }
    template <int SLICES, typename Beside>
    __device__ __forceinline__ void run(const f32x16& p, const float (&scale)[SLICES], f32x16 (&acc)[NB], Beside&& beside) {
        Parts b[2];
        auto split = [&](auto s) {
            // (register r holds row 8 * (r / 4) + 4 * h + r % 4: four registers, eight rows)
            i32x2 h0, l0, h1, l1;
            split_quad(p[8 * s], p[8 * s + 1], p[8 * s + 2], p[8 * s + 3], scale[2 * s * SLICES / 4], h0, l0);
            split_quad(p[8 * s + 4], p[8 * s + 5], p[8 * s + 6], p[8 * s + 7], scale[(2 * s + 1) * SLICES / 4], h1, l1);
            b[s] = Parts{{h0[0], h0[1], h1[0], h1[1]}, {l0[0], l0[1], l1[0], l1[1]}};
        };
        split(std::integral_constant<int, 0>{});
        static_for<N>([&](auto u) {
            acc[u % NB] = mma_parts(a[u], b[u / NB], acc[u % NB]);
            if constexpr (u == 0) split(std::integral_constant<int, 1>{});  // the second half of P under the first MFMAs
            read<u + AHEAD>();
            beside(u);
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    template <int SLICES>
    __device__ __forceinline__ void run(const f32x16& p, const float (&scale)[SLICES], f32x16 (&acc)[NB]) {
        run(p, scale, acc, [](auto) {});
    }
};

template <int N>
__device__ __forceinline__ void scale_blocks(f32x16 (&x)[N], float f) {
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) x[i][r] *= f;
}
// x * 2^e (any e)
template <int N>
__device__ __forceinline__ void ldexp_blocks(f32x16 (&x)[N], int e) {
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) x[i][r] = __builtin_amdgcn_ldexpf(x[i][r], e);
}

// The common scale of a sum over blocks, X_1^T Y_1 + X_2^T Y_2 + ...: X of a block comes in slices of rows with the field of
// their scales, Y is a 32x32 block of which every lane scales its own column.
// Probabilities, at most 1, are scaled to 2^15 against the smallest X field so far.
struct ProbabilitySum {
    int ref = kPartsHigh;  // the smallest field so far (the same in every lane)
    template <int N, int SLICES>
    __device__ __forceinline__ void scales(const int (&field)[SLICES], f32x16 (&acc)[N], float (&out)[SLICES]) {
        int least = field[0];
#pragma unroll
        for (int i = 1; i < SLICES; i++) least = imin(least, field[i]);
        if (least < ref) {
            scale_blocks(acc, pow2_of_field(127 + least - ref));
            ref = least;
        }
#pragma unroll
        for (int i = 0; i < SLICES; i++) out[i] = pow2_of_field(127 + 15 + ref - field[i]);
    }
    template <int N>
    __device__ __forceinline__ void finish(f32x16 (&acc)[N]) const {
        ldexp_blocks(acc, 127 - 15 - ref);
    }
};
// Score gradients: scaled by the running maximum of the lane's column (both halves), with two bits of room so that the sums are
// rescaled rarely.
struct GradientSum {
    int ref = kPartsHigh, column = kPartsHigh;
    template <int N, int SLICES>
    __device__ __forceinline__ void scales(const f32x16& y, const int (&field)[SLICES], f32x16 (&acc)[N], float (&out)[SLICES]) {
        float m = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r += 2) m = max3_abs(m, y[r], y[r + 1]);
        const int col = parts_field(max_bits_across_halves(max_bits(m)));
        const bool grow = col < column;
        int least = field[0];
#pragma unroll
        for (int i = 1; i < SLICES; i++) least = imin(least, field[i]);
        if (least < ref || __builtin_amdgcn_ballot_w64(grow) != 0) {
            const int column_new = grow ? col - 2 : column, ref_new = imin(least, ref);
            scale_blocks(acc, pow2_of_field(127 + column_new - column + ref_new - ref));
            column = column_new;
            ref = ref_new;
        }
#pragma unroll
        for (int i = 0; i < SLICES; i++) out[i] = pow2_of_field(column + ref - field[i]);
    }
    template <int N>
    __device__ __forceinline__ void finish(f32x16 (&acc)[N]) const {
        ldexp_blocks(acc, 254 - column - ref);
    }
};

// 0 where every register of the blocks is finite in this lane, NaN otherwise
template <int N>
__device__ __forceinline__ float finite_probe(const f32x16 (&x)[N], float acc) {
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc = __builtin_fmaf(x[i][r], 0.f, acc);
    return acc;
}

}  // namespace chill
