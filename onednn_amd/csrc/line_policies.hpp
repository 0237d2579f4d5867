// Operand policies of the whole-line loops (line_loops.hpp):
//   acc_t, NU       accumulator of a 16 x 16 tile, instructions of a fragment pair and step
//   SCALE_SETS      sets of four block scales of a step, 0 = no block scales
//   SCALED, FULL    for the chain kernels: src and weights scales are the epilogue's; every activation is carried
//   prepare_a / b   what a fragment needs before its first product
//   mma<J, I>       instruction u of a pair; J, I = column tile and row tile inside a half, which pick scale bytes
//   mma_tied        the same as inline assembly, accumulator tied
// The MFMA operands are exchanged (weights first): the tile comes out transposed, a lane holds four consecutive n of
// one row.
#pragma once
#include "line_loops.hpp"

namespace mi355 {
namespace {

using namespace gemm;
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));
typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));

// bf16 (BF16) or f16 operands on the 16 x 16 x 32 instruction, in the whole-line loops.  The 32 x 32 x 16 shape costs
// the same matrix cycles and LDS bytes but sustains 1.53 instead of 1.85 PFLOP/s on random operand bits (the clock the
// power manager allows, `bench.py --calib-mfma`).
template <bool BF16, class G_>
struct h16x16_mma_t {
    using G = G_;
    static constexpr bool TILE16 = true;
    static constexpr int ELEM_BYTES = 2;
    static constexpr int ROWS = 8, COLS = G::WCOLS / 16;
    static constexpr int NU = 2, SCALE_SETS = 0;
    typedef v4f acc_t;
    static constexpr bool SCALED = false, INTEGER = false, FULL = true;
    __device__ static __forceinline__ void prepare_a(line_pair_t &) {}
    __device__ static __forceinline__ void prepare_b(line_pair_t &) {}
    // operands exchanged: the tile comes out transposed (a lane holds four consecutive n of one row)
    template <int, int, class U>
    __device__ static __forceinline__ void mma(v4f &acc, const line_pair_t &b, const line_pair_t &a, U, int, int) {
        constexpr int u = U::value;
        if constexpr (BF16)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_t, b.c[u]), __builtin_bit_cast(v8bf_t, a.c[u]),
                    acc, 0, 0, 0);
        else
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h_t, b.c[u]), __builtin_bit_cast(v8h_t, a.c[u]),
                    acc, 0, 0, 0);
    }
    template <int, int>
    __device__ static __forceinline__ void mma_tied(v4f &acc, const line_pair_t &b, const line_pair_t &a, int u, int, int) {
        if constexpr (BF16)
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(b.c[u]), "v"(a.c[u]));
        else
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b.c[u]), "v"(a.c[u]));
    }
};

// the same for a dst of the other 16-bit type: chains without the activations that take a hardware exponential
template <bool BF16, class G_>
struct h16_mixed_mma_t : h16x16_mma_t<BF16, G_> {
    static constexpr bool FULL = false;
};

// the same with the weights (ACROSS = 1), or src and the weights (2), contiguous across K
template <bool BF16, class G_, int ACROSS>
struct h16_across_mma_t : h16x16_mma_t<BF16, G_> {
    static constexpr bool A_KM = ACROSS == 2, B_KM = true;
};

// int8 on v_mfma_i32_16x16x64_i8 (sustains ~4.0 POPS on this hardware, the 32 x 32 x 32 shape ~3.0).  u8 operands are
// re-biased to s8 in registers; bytes beyond K are zeroed after that.
template <bool SRC_U8, bool WEI_U8, class G_>
struct i8_mma_t {
    using G = G_;
    static constexpr int ROWS = 8, COLS = G::WCOLS / 16;
    static constexpr int NU = 2, SCALE_SETS = 0;
    typedef v4i acc_t;
    static constexpr bool SCALED = true, INTEGER = true, FULL = false;
    __device__ static __forceinline__ void flip(line_pair_t &f) {
#pragma unroll
        for (int u = 0; u < 2; ++u) f.c[u] ^= (int)0x80808080;
    }
    __device__ static __forceinline__ void prepare_a(line_pair_t &f) {
        if (SRC_U8) flip(f);
    }
    __device__ static __forceinline__ void prepare_b(line_pair_t &f) {
        if (WEI_U8) flip(f);
    }
    template <int, int, class U>
    __device__ static __forceinline__ void mma(v4i &acc, const line_pair_t &b, const line_pair_t &a, U, int, int) {
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(b.c[U::value], a.c[U::value], acc, 0, 0, 0);
    }
    template <int, int>
    __device__ static __forceinline__ void mma_tied(v4i &acc, const line_pair_t &b, const line_pair_t &a, int u, int, int) {
        asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(acc) : "v"(b.c[u]), "v"(a.c[u]));
    }
};

// fp8 on v_mfma_f32_16x16x128_f8f6f4, one instruction a pair (registers only, random operand bits: 4.9 PFLOP/s against 4.5
// of the 32 x 32 x 64 shape).  FMT: 0 = e4m3, 1 = e5m2.  Where a byte of K sits inside the instruction does not matter
// without block scales, both operands hold it in the same place.
template <int FMT_A, int FMT_B, class G_>
struct f8_mma_t {
    using G = G_;
    static constexpr bool TILE16 = true;
    static constexpr int ELEM_BYTES = 1;
    static constexpr int ROWS = 8, COLS = G::WCOLS / 16;
    static constexpr int NU = 1, SCALE_SETS = 0;
    typedef v4f acc_t;
    static constexpr bool SCALED = true, INTEGER = false, FULL = true;
    __device__ static __forceinline__ void prepare_a(line_pair_t &) {}
    __device__ static __forceinline__ void prepare_b(line_pair_t &) {}
    template <int, int, class U>
    __device__ static __forceinline__ void mma(v4f &acc, const line_pair_t &b, const line_pair_t &a, U, int, int) {
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b.whole(), a.whole(), acc, FMT_B, FMT_A, 0, 0, 0, 0);
    }
    template <int, int>
    __device__ static __forceinline__ void mma_tied(v4f &acc, const line_pair_t &b, const line_pair_t &a, int, int, int) {
        const v8i B = b.whole(), A = a.whole();
        asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:%3 blgp:%4"
                     : "+a"(acc)
                     : "v"(B), "v"(A), "n"(FMT_B), "n"(FMT_A));
    }
};

// MXFP8: the same with e8m0 scales per 32 k of both operands, applied by the instruction.  With scales the placement of K
// counts: the instruction reads the first register halves of the lane groups 0 .. 3 (16 lanes each) as k 0..63, 16 each,
// the second halves as k 64..127, and takes the scale of block g (k 32 g .. 32 g + 31) from lane group g -- the
// fragments' own order and the packed scales'.
template <int FMT_A, int FMT_B, class G_>
struct mxf8_mma_t : f8_mma_t<FMT_A, FMT_B, G_> {
    static constexpr bool MX = true;
    static constexpr int SCALE_SETS = 1;
    static constexpr bool SCALED = false;
    template <int J, int I, class U>
    __device__ static __forceinline__ void mma(v4f &acc, const line_pair_t &b, const line_pair_t &a, U, int sb, int sa) {
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b.whole(), a.whole(), acc, FMT_B, FMT_A, J, sb, I, sa);
    }
    // (the scale's byte: op_sel its bit 0, op_sel_hi its bit 1)
    template <int J, int I>
    __device__ static __forceinline__ void mma_tied(v4f &acc, const line_pair_t &b, const line_pair_t &a, int, int sb, int sa) {
        const v8i B = b.whole(), A = a.whole();
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[%5,%6,0] op_sel_hi:[%7,%8,0] cbsz:%9 blgp:%10"
                     : "+a"(acc)
                     : "v"(B), "v"(A), "v"(sb), "v"(sa), "n"(J & 1), "n"(I & 1), "n"(J >> 1), "n"(I >> 1), "n"(FMT_B), "n"(FMT_A));
    }
};

// MXFP4: 64 bytes of K are the 128 k of one v_mfma_scale_f32_16x16x128_f8f6f4, four blocks of 32; lane group g supplies
// block g and its scale.  (The order of the two nibbles of a byte does not matter: both operands agree, and the 32
// elements of a block share one scale.)
template <class G_>
struct mxf4_mma_t {
    using G = G_;
    static constexpr bool MX = true;
    static constexpr int ROWS = 8, COLS = G::WCOLS / 16;
    static constexpr int NU = 2, SCALE_SETS = 2;
    typedef v4f acc_t;
    static constexpr bool SCALED = false, INTEGER = false, FULL = false;
    __device__ static __forceinline__ void prepare_a(line_pair_t &) {}
    __device__ static __forceinline__ void prepare_b(line_pair_t &) {}
    template <int J, int I, class U>
    __device__ static __forceinline__ void mma(v4f &acc, const line_pair_t &b, const line_pair_t &a, U, int sb, int sa) {
        const v4i &x = b.c[U::value], &y = a.c[U::value];
        acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(v8i {x[0], x[1], x[2], x[3], 0, 0, 0, 0},
                v8i {y[0], y[1], y[2], y[3], 0, 0, 0, 0}, acc, 4, 4, J, sb, I, sa);
    }
    template <int J, int I>
    __device__ static __forceinline__ void mma_tied(v4f &acc, const line_pair_t &b, const line_pair_t &a, int u, int sb, int sa) {
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[%5,%6,0] op_sel_hi:[%7,%8,0] cbsz:4 blgp:4"
                     : "+a"(acc)
                     : "v"(b.c[u]), "v"(a.c[u]), "v"(sb), "v"(sa), "n"(J & 1), "n"(I & 1), "n"(J >> 1), "n"(I >> 1));
    }
};

} // namespace
} // namespace mi355
