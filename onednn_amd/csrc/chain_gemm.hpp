// GEMM kernels whose epilogue is compiled in: the K loops of line_loops.hpp, then one of the chains that layers are
// made of,
//   f32(acc [+ compensation[n]]) [* src_scale * wei_scale[n]] [+ bias[n]] [-> relu | gelu_tanh | swish]
//       [+ or * bf16 tensor] [/ dst_scale] -> bf16 / f16 / f32 / s8 / u8
// The families' general kernels (tile_epilogue.hpp) decide all of that at run time from the problem's description, in
// 400 KB of code that a workgroup runs through once: 13 us after every tile for a bias and a bf16 dst, most of it
// instruction fetches.  Here the host decides (chain_from), the arguments are what the chain uses, and a tile's epilogue
// is a straight run of a few KB.
//
// Global memory sees whole rows of the wavefront's 128 x 64 part.  In the accumulator layout a wavefront-wide store
// touches 16 rows, 4 to 16 bytes a lane of each, and the memory pipeline's cost is per piece of a line; so the part
// goes through the wavefront's 16 KB share of the idle ring and leaves 1 KB a store.  LDS rows are 64 / 128 / 256 bytes for
// 1- / 2- / 4-byte elements, the 16-byte chunks of a row XOR-swizzled so that neither the writes (16 rows, the same
// columns) nor the reads (whole rows) meet on a bank; 4-byte elements leave in two passes of 64 rows.  The bf16 tensor
// of the chain comes the other way, all of it in flight at once, and a quad of it is read from the cell that its result
// is written to.
#pragma once
#include "line_loops.hpp"

namespace mi355 {

enum chain_dst_t { CHAIN_BF16, CHAIN_F16, CHAIN_F32, CHAIN_I8, CHAIN_PART }; // CHAIN_PART: a part of K, no epilogue
enum chain_act_t { CHAIN_NONE, CHAIN_RELU, CHAIN_GELU, CHAIN_SWISH };

// Into how many parts of K a problem of few tiles is split, 1 = not at all.  One workgroup a CU and round: with T tiles
// (256 x 128, or 256 x 256) a launch takes its K steps one after the other on T of 256 CUs.  S parts make that steps / S, for
// a second kernel (3 us and more of a launch), the parts' way out and in again (a part of a tile 128 / 256 KB each way) and
// a workgroup's fixed cost, which is why S is not 256 / T: per step_ns + S T part_ns + CHAIN_SPLIT_NS is what a launch of S
// parts of `per` steps takes beyond one without.  Its S against the best of up to 12 on 22 shapes of every type: within 1.05 on
// 18, at worst 1.15 (fp8 300 x 2048 x 2048, which it does not split: 17.4 us, two parts 15.1).  Unsplit / split, us, launches after each
// other on the same operands: fp8 256 x 4352 x 12224 73.8 / 27.8, 64 x 640 x 16384 67.3 / 15.8, 512 x 7168 x 16384 (two parts) 74.5 / 59.0; MXFP4
// 100 x 1040 x 16352 55.0 / 23.3; bf16 4096 x 960 x 13312 118 / 92.9, f16 300 x 2048 x 4096 39.2 / 19.6; int8 256 x 6272 x 6528 (u8) 50.6 /
// 34.9; where steps are few the second kernel costs more than it gives (bf16 512 x 3600 x 704 14.8 / 19.2 in two parts).
constexpr long CHAIN_SPLIT_NS = 5000;
struct chain_split_t {
    int split, part_steps;
};
inline chain_split_t chain_split(long batch, long M, long N, long kbytes, bool wide, long step_ns) {
    const long bn = wide ? 256 : 128, tiles = batch * ((M + 255) / 256) * ((N + bn - 1) / bn), steps = (kbytes + 127) / 128;
    const long part_ns = wide ? 104 : 52;
    chain_split_t r {1, (int)steps};
    if (tiles < 1 || tiles > 128) return r;
    long best = steps * step_ns - CHAIN_SPLIT_NS;
    // (no s does better than the least of steps / s * step_ns + s * tiles * part_ns: most launches leave here)
    if (best <= 0 || 4. * steps * step_ns * tiles * part_ns >= (double)best * best) return r;
    for (long s = 2; s * tiles <= 256; ++s) {
        const long per = (steps + s - 1) / s;
        if (per < 2) break;
        if ((steps + per - 1) / per != s) continue; // (the same steps a part with fewer of them)
        const long ns = per * step_ns + s * tiles * part_ns;
        if (ns < best) best = ns, r = chain_split_t {(int)s, (int)per};
    }
    return r;
}
inline size_t chain_parts_bytes(long batch, long M, long N, bool wide, int split) {
    const long bn = wide ? 256 : 128;
    return split > 1 ? (size_t)(batch * ((M + 255) / 256) * ((N + bn - 1) / bn)) * split * (size_t)(256 * bn * 4) : 0;
}

struct chain_vec_t { // f32 / bf16 / f16 values; dt UNDEF = absent
    const void *p;
    int dt, per; // per: one value for every column (weights scales, bias) or row (src scales) instead of one for all
    long bs;     // elements between batches
};

struct chain_t {
    const char *a, *bt;
    char *dst;
    long lda, ldb, a_bs, b_bs, dst_pitch, dst_bs; // bytes
    long M, N, kbytes;
    int tiles_m, tiles_n;
    gemm::line_scales_args_t sc;
    chain_vec_t ssc, wsc, bias;
    int act, staged; // staged: 1 = + the bf16 tensor, 2 = * it
    float alpha;
    const char *st;
    long st_pitch, st_bs;
    // int8: (K sum) + (off_s - src zero point) * colsum[n]
    const int *colsum, *src_zp;
    long colsum_bs;
    int off_s;
    const void *dsc;
    int dsc_dt, ds_mode; // 0 none, 1 divide, 2 multiply by the reciprocal
    int lo, hi;          // 8-bit dst
};

// ... and what the kernels of parts of K and of the 32 x 32 tiles of 16-bit, fp8 and block-scaled operands also read; a type of
// its own, so that the others' arguments are no longer for it (every launch writes them to the device)
struct chain_more_t : chain_t {
    // split > 1: K in parts of part_steps steps, a workgroup each; their accumulators go to parts and chain_sum_kernel
    // (kern_chain_sum.hip) adds them and does the rest
    char *parts;
    int split, part_steps;
    // e8m0 scales as the caller has them (chain_launch_small): [M][K / 32] and [K / 32][N], values between batches
    const uint8_t *sa, *sb;
    long sa_bs, sb_bs;
};
template <int DST>
using chain_arg_t = std::conditional_t<DST == CHAIN_PART, chain_more_t, chain_t>; // of chain_gemm_kernel

// A product of few 32 x 32 tiles on chain_small_float_kernel (kern_chain_small.hip): small_tiles_float says whether (mx: 0, or
// the bits of a block-scaled type).
enum chain_small_t { CHAIN_SMALL_BF16, CHAIN_SMALL_F16, CHAIN_SMALL_F8, CHAIN_SMALL_MXF8, CHAIN_SMALL_MXF4 };
// small_tiles_fit: whether its 32-bit steps of K and offsets of block scales reach that far.
bool small_tiles_fit(long M, long N, long kbytes, int mx);
bool small_tiles_float(long batch, long M, long N, long kbytes, const chain_split_t &split, long step_ns, const chain_t &C, int mx);
int chain_launch_small(chain_small_t kind, int dst_dt, chain_more_t &C, unsigned batch, hipStream_t stream);

// the sums of a problem whose parts lie at C.parts, and its epilogue (integer: they are s32)
int chain_launch_sum(bool integer, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream);

// The problem's epilogue as a chain; false: not one of them (the general kernels run it).  What the K loop reads (a,
// bt, lda, ldb, the batches' strides, kbytes, block scales, colsum) is the family's to fill in.  scaled: src and
// weights scales are the epilogue's; full: activations other than relu and the bf16 tensor are carried.
bool chain_from(const problem_t &P, bool scaled, bool full, chain_t &C);
// ... in two parts: what the descriptor decides (problem_of_desc, kernels.hpp, is enough of a problem), and whether dst lies
// where whole pieces of its rows can be stored
bool chain_form(const problem_t &P, bool scaled, bool full, chain_t &C);
inline bool chain_dst_aligned(const chain_t &C, int dst_dt) { return ((uintptr_t)C.dst & (dt_bits(dst_dt) == 8 ? 3 : 15)) == 0; }

// the same for a family with block scales: where mx is set they are operands of the instruction
bool chain_from_mx(const problem_t &P, bool mx, bool full, chain_t &C);

// mx_pack_scales (kern_mxf4.hip): the pre-pass of the block-scaled types
int mx_pack_scales(const mi355_matmul_desc_t &d, const problem_t &P, long Bsa, long Bsb, char *sa, char *sb,
        gemm::line_scales_args_t &sc, hipStream_t stream);

// The families' launchers on the chain kernels, a translation unit each; C as chain_from and the family left it.
// wide: the 256 x 256 tiles whatever the size.  A 16-bit dst of the operands' other type takes a C of full = false.
int chain_launch_h16(bool bf16, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream);
// ... with the weights (across = 1), or src and the weights (2, 256 x 256 tiles only), contiguous across K: lda / ldb are the
// bytes from one k to the next
int chain_launch_h16_across(bool bf16, int dst_dt, int across, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream);
int chain_launch_i8(bool src_u8, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream);
// ... on 32 x 32 tiles that make their own column sums (C.colsum is not read)
int chain_launch_i8_small(bool src_u8, int dst_dt, chain_t &C, unsigned batch, hipStream_t stream);
int chain_launch_f8(int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream); // e4m3 x e4m3
int chain_launch_mx(bool fp4, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream); // e4m3 x e4m3 or fp4

#ifdef MI355_CHAIN_KERNELS
namespace {
using namespace gemm;

__device__ __forceinline__ float chain_load(const chain_vec_t &v, long i) {
    if (v.dt == MI355_DT_F32) return ((const float *)v.p)[i];
    const uint16_t h = ((const uint16_t *)v.p)[i];
    return v.dt == MI355_DT_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
}

typedef unsigned v2u_cell_t __attribute__((ext_vector_type(2)));
typedef unsigned v4u_cell_t __attribute__((ext_vector_type(4)));
typedef unsigned __attribute__((address_space(3), may_alias)) *lds_cell1_t;
typedef v2u_cell_t __attribute__((address_space(3), may_alias)) *lds_cell2_t;
typedef v4u_cell_t __attribute__((address_space(3), may_alias)) *lds_cell4_t;

// LDS rows of the part; SHIFT = log2 of the element's bytes
template <int SHIFT>
__device__ __forceinline__ int cell_swizzle(int r) {
    return SHIFT == 0 ? (r >> 2) & 3 : SHIFT == 1 ? (r >> 1) & 7 : r & 15;
}
// the lane's four columns 16 k + 4 (lane / 16) of row r
template <int SHIFT>
__device__ __forceinline__ unsigned cell_of(unsigned part, int r, int k, int lane) {
    const int at = (16 * k + 4 * (lane >> 4)) << SHIFT;
    const int row = SHIFT == 2 ? r & 63 : r;
    return part + (unsigned)((row << (6 + SHIFT)) + (((at >> 4) ^ cell_swizzle<SHIFT>(r)) << 4) + (at & 15));
}

// Rows r0 .. r0 + COUNT - 1 of the part to dst.  (A wavefront reads back what its own lanes wrote: program order, no
// barrier.)  cols_left: columns of dst from the part's first one on.
template <int SHIFT, int COUNT>
__device__ __forceinline__ void flush_rows(unsigned part, char *base, long pitch, int r0, long rows_left, long cols_left,
        int lane) {
    constexpr int LANES = 4 << SHIFT, ROWS = 64 / LANES, PER = 16 >> SHIFT; // lanes a row, rows a store, columns a lane
    const int slot = lane & (LANES - 1);
    // (a uniform test: a pitch or base that is not 16-byte aligned, 8-bit dst only, leaves in dwords)
    const bool pieces = SHIFT == 0 && (((uintptr_t)base | (uintptr_t)pitch) & 15) != 0;
#pragma unroll
    for (int d = 0; d < COUNT / ROWS; ++d) {
        const int r = r0 + d * ROWS + lane / LANES;
        const v4u_cell_t q = *(lds_cell4_t)(size_t)(part + (unsigned)(d * 1024 + lane * 16));
        const int col = (slot ^ cell_swizzle<SHIFT>(r)) * PER;
        char *to = base + r * pitch + (col << SHIFT);
        if (r >= rows_left || col >= cols_left) continue;
        if (col + PER <= cols_left && !pieces) {
            // whole lines, written once and not read again by this launch: non-temporal
            if (SHIFT == 0) *(v4u_cell_t *)to = q;
            else __builtin_nontemporal_store(q, (v4u_cell_t *)to);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = col + e * (4 >> SHIFT);
                if (c + (4 >> SHIFT) <= cols_left) {
                    *(unsigned *)(to + 4 * e) = q[e];
                } else if (SHIFT == 1 && c < cols_left) {
                    *(uint16_t *)(to + 4 * e) = (uint16_t)q[e];
                } else if (SHIFT == 0) {
#pragma unroll
                    for (int x = 0; x < 3; ++x)
                        if (c + x < cols_left) to[4 * e + x] = (char)(q[e] >> (8 * x));
                }
            }
        }
    }
}

// bf16 of four values: v_cvt_pk_bf16_f32 is the reference's rounding for normal numbers, zeros and infinities; the
// reference flushes f32 subnormals and quiets NaNs its own way, so a wavefront that holds either converts in software
__device__ __forceinline__ v2u_cell_t chain_bf16(const float (&x)[4], bool soft) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    if (__builtin_expect(soft, 0))
        return v2u_cell_t {f32_to_bf16(x[0]) | ((unsigned)f32_to_bf16(x[1]) << 16),
                f32_to_bf16(x[2]) | ((unsigned)f32_to_bf16(x[3]) << 16)};
    return v2u_cell_t {__builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t {x[0], x[1]}, bf16x2_t)),
            __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2_t {x[2], x[3]}, bf16x2_t))};
}

// The per-column table of a workgroup: scale, bias, compensation of its columns, 256 each
constexpr int CT_WSC = 0, CT_BIAS = 1, CT_COMP = 2, CT_BYTES = 3 * 256 * 4;

template <class Mma>
struct chain_part_t {
    const chain_t &C;
    unsigned tab, part;
    long b, m_base, n_base;
    int lane, col0;
    float ds, ds_inv;
    int ds_mode; // 0 none, 1 divide, 2 multiply by the reciprocal, 3 divide by fma correction

    __device__ __forceinline__ v4f tab4(int slot, int k) const {
        typedef const v4f __attribute__((address_space(3))) *lds_v4f_t;
        return *(lds_v4f_t)(size_t)(tab + (unsigned)((slot * 256 + col0 + 16 * k + 4 * (lane >> 4)) * 4));
    }
    // STAGED: the chain may have a bf16 tensor
    template <int DST, int ACT, bool STAGED, class V>
    __device__ __forceinline__ void store(const V (&acc)[8][4]) const {
        constexpr int SHIFT = DST == CHAIN_I8 ? 0 : DST == CHAIN_F32 ? 2 : 1;
        const bool staged = STAGED && C.staged;
        const int lrow = lane & 15;
        const long rows_left = C.M - m_base, cols_left = C.N - n_base;
        if (rows_left <= 0 || cols_left <= 0) return;
        char *base = C.dst + b * C.dst_bs + m_base * C.dst_pitch + (n_base << SHIFT);
        if (staged) {
            const char *from = scalar_ptr(C.st + b * C.st_bs + m_base * C.st_pitch + n_base * 2);
            // (columns in whole chunks, chain_from; those beyond N repeat the last chunk, rows beyond M the last row)
            const int last = (int)(cols_left < 64 ? cols_left : 64) / 8 - 1;
#pragma unroll
            for (int d = 0; d < 16; ++d) {
                const int r = d * 8 + (lane >> 3), chunk = min((lane & 7) ^ cell_swizzle<1>(r), last);
                const long rv = r < rows_left ? r : rows_left - 1;
                dma16(from, (unsigned)(rv * C.st_pitch + chunk * 16), part + (unsigned)d * 1024u);
            }
        }
        v4f w[4], bb[4];
        v4i comp[4];
        float ssc = 1.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (Mma::SCALED) w[k] = tab4(CT_WSC, k);
            bb[k] = tab4(CT_BIAS, k);
            if (Mma::INTEGER) comp[k] = __builtin_bit_cast(v4i, tab4(CT_COMP, k));
        }
        const bool bias = C.bias.dt != MI355_DT_UNDEF;
        if (Mma::SCALED && C.ssc.dt != MI355_DT_UNDEF && !C.ssc.per) ssc = chain_load(C.ssc, b * C.ssc.bs);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 16 * i + lrow;
            if (Mma::SCALED && C.ssc.per) ssc = chain_load(C.ssc, b * C.ssc.bs + m_base + (r < rows_left ? r : rows_left - 1));
            if (staged) {
                wait_vmcnt_upto(14 - 2 * i); // the two loads of this row block have landed
                asm volatile("" ::: "memory"); // no LDS read moves above the wait
            }
            float x[4][4];
            bool special = false;
            unsigned mag = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float t;
                    if constexpr (Mma::INTEGER) t = (float)(acc[i][k][e] + comp[k][e]);
                    else t = acc[i][k][e];
                    if (Mma::SCALED) t *= ssc, t *= w[k][e];
                    x[k][e] = t;
                }
            }
            if (bias) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[k][e] += bb[k][e];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float t = x[k][e];
                    if (ACT == CHAIN_RELU) {
                        if (DST == CHAIN_I8) t = fmaxf(t, 0.f); // an integer dst turns NaN and -0 into 0 either way
                        else t = t > 0 ? t : t * 0.f;
                    } else if (ACT == CHAIN_GELU) {
                        t = gelu_tanh_fast(t);
                    } else if (ACT == CHAIN_SWISH) {
                        t = t * logistic_fast(C.alpha * t);
                    }
                    x[k][e] = t;
                }
            if (staged) {
                const bool add = C.staged == 1;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const v2u_cell_t q = *(lds_cell2_t)(size_t)cell_of<1>(part, r, k, lane);
                    const float y[4] = {u2f(q.x << 16), u2f(q.x & 0xffff0000u), u2f(q.y << 16), u2f(q.y & 0xffff0000u)};
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[k][e] = add ? x[k][e] + y[e] : x[k][e] * y[e];
                }
            }
            if constexpr (DST == CHAIN_I8) {
                if (ds_mode & 1) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
#pragma unroll
                        for (int e = 0; e < 4; ++e) mag = max(mag, mag_bits(x[k][e]));
                    if (ds_mode == 3 && __builtin_expect(__builtin_amdgcn_ballot_w64(mag >= DIV_BY_FMA_LIMIT) == 0, 1)) {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[k][e] = div_by_fma(x[k][e], ds, ds_inv);
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[k][e] /= ds;
                    }
                } else if (ds_mode == 2) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[k][e] *= ds_inv;
                }
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    *(lds_cell1_t)(size_t)cell_of<0>(part, r, k, lane) = pack4_i8(x[k], C.lo, C.hi);
            } else if constexpr (DST == CHAIN_F32) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    *(lds_cell4_t)(size_t)cell_of<2>(part, r, k, lane)
                            = v4u_cell_t {f2u(x[k][0]), f2u(x[k][1]), f2u(x[k][2]), f2u(x[k][3])};
                if (i == 3) flush_rows<2, 64>(part, base, C.dst_pitch, 0, rows_left, cols_left, lane);
            } else if constexpr (DST == CHAIN_F16) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    unsigned h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) h[e] = __builtin_bit_cast(uint16_t, (_Float16)x[k][e]);
                    *(lds_cell2_t)(size_t)cell_of<1>(part, r, k, lane) = v2u_cell_t {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) special |= __builtin_amdgcn_classf(x[k][e], 0x93); // NaN or subnormal
                const bool soft = __builtin_amdgcn_ballot_w64(special) != 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) *(lds_cell2_t)(size_t)cell_of<1>(part, r, k, lane) = chain_bf16(x[k], soft);
            }
        }
        if (DST == CHAIN_F32) flush_rows<2, 64>(part, base, C.dst_pitch, 64, rows_left, cols_left, lane);
        else flush_rows<SHIFT, 128>(part, base, C.dst_pitch, 0, rows_left, cols_left, lane);
    }
    // (n is a constant after unrolling)
    __device__ __forceinline__ static void wait_vmcnt_upto(int n) {
        switch (n) {
            case 14: wait_vmcnt<14>(); break;
            case 12: wait_vmcnt<12>(); break;
            case 10: wait_vmcnt<10>(); break;
            case 8: wait_vmcnt<8>(); break;
            case 6: wait_vmcnt<6>(); break;
            case 4: wait_vmcnt<4>(); break;
            case 2: wait_vmcnt<2>(); break;
            default: wait_vmcnt<0>(); break;
        }
    }
};

extern __shared__ __attribute__((aligned(128))) char chain_smem[];

template <class Mma, int DST>
__global__ void __launch_bounds__(Mma::G::NT) __attribute__((amdgpu_waves_per_eu(Mma::G::NW / 4))) chain_gemm_kernel(const chain_arg_t<DST> C) {
    using G = typename Mma::G;
    using V = typename Mma::acc_t;
    static_assert(G::WCOLS == 64, "a wavefront's part is 128 x 64");
    char *smem = chain_smem;
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    constexpr bool PART = DST == CHAIN_PART;
    long b = blockIdx.z, step0 = 0; // (the first step of the part)
    if constexpr (PART) {
        b = blockIdx.z / C.split;
        step0 = (long)(blockIdx.z % C.split) * C.part_steps;
    }
    const tile_pos_t tp = tile_position<G>((int)blockIdx.x, C.tiles_m, C.tiles_n);
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;
    const unsigned tab = lds0 + line_loader_t<Mma>::LDS_BYTES;
    auto fill = [&]() __attribute__((always_inline)) {
        if constexpr (PART) return;
        typedef int __attribute__((address_space(3))) *lds_i_t;
        static_assert(G::NT % 256 == 0, "every column has a thread");
        const int col = t & 255;
        const long n = tp.n0 + col < C.N ? tp.n0 + col : C.N - 1;
        lds_i_t at = (lds_i_t)(size_t)(tab + (unsigned)(col * 4));
        if (Mma::SCALED)
            at[CT_WSC * 256] = __float_as_int(C.wsc.dt != MI355_DT_UNDEF ? chain_load(C.wsc, b * C.wsc.bs + (C.wsc.per ? n : 0)) : 1.f);
        if (C.bias.dt != MI355_DT_UNDEF) at[CT_BIAS * 256] = __float_as_int(chain_load(C.bias, b * C.bias.bs + n));
        if (Mma::INTEGER) {
            const int a = C.off_s - (C.src_zp ? *C.src_zp : 0);
            at[CT_COMP * 256] = C.colsum ? a * C.colsum[b * C.colsum_bs + n] : 0;
        }
    };
    V acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = V {0, 0, 0, 0};
    line_scales_t sc = C.sc.tile(b, tp.m0, tp.n0);
    long kbytes = C.kbytes;
    if constexpr (PART) {
        kbytes = min(kbytes - step0 * LKB, (long)C.part_steps * LKB);
        sc.a += step0 * Mma::SCALE_SETS * sc.a_pitch;
        sc.b += step0 * Mma::SCALE_SETS * sc.b_pitch;
        sc.sets -= (int)step0 * Mma::SCALE_SETS;
    }
    main_loop_lines<Mma>(acc, smem,
            C.a + b * C.a_bs + (line_form<Mma>::AKM ? tp.m0 * 2 + step0 * 64 * C.lda : tp.m0 * C.lda + step0 * LKB),
            C.bt + b * C.b_bs + (line_form<Mma>::BKM ? tp.n0 * 2 + step0 * 64 * C.ldb : tp.n0 * C.ldb + step0 * LKB), C.lda, C.ldb,
            C.M - tp.m0, C.N - tp.n0, kbytes, sc, fill);
    if constexpr (PART) { // [part][tile][wavefront][accumulator quad][lane]
        char *to = C.parts + (((long)blockIdx.z * gridDim.x + blockIdx.x) * G::NW + wave) * 32768 + (t & 63) * 16;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) *(V *)(to + (i * 4 + j) * 1024) = acc[i][j];
        return;
    } else {

    const int wm = G::wm(wave), wn = G::wn(wave);
    chain_part_t<Mma> E {C, tab, lds0 + (unsigned)wave * 16384u, b, tp.m0 + wm * 128, tp.n0 + wn * 64, t & 63, wn * 64, 1.f, 1.f, 0};
    if (DST == CHAIN_I8 && C.ds_mode != 0) {
        E.ds = chain_load(chain_vec_t {C.dsc, C.dsc_dt, 0, 0}, 0);
        E.ds_inv = 1.f / E.ds;
        // division by fma correction where its proof holds (tile_epilogue.hpp); a mode of 1 divides
        const float as = fabsf(E.ds);
        E.ds_mode = C.ds_mode == 2 ? 2 : as >= 0x1p-20f && as <= 0x1p20f ? 3 : 1;
    }
    constexpr bool FULL = DST != CHAIN_I8 && DST != CHAIN_F32 && Mma::FULL;
    // A launch of few steps is bound by its epilogue's instruction fetches, and the second tensor's code is in the way of a
    // chain without one: the 16-bit types have both (1 x 512 x 64, bf16: 9.4 -> 8.4 us).  fp8's scales leave no registers
    // for that (4096 x 28672 x 8192 with gelu and residual: 706 -> 723 us, 72 bytes a lane in scratch memory).
    constexpr bool BOTH = FULL && !Mma::SCALED && Mma::SCALE_SETS == 0;
    auto store = [&](auto staged) __attribute__((always_inline)) {
        constexpr bool S = decltype(staged)::value;
        if constexpr (FULL) {
            if (C.act == CHAIN_GELU) return E.template store<DST, CHAIN_GELU, S>(acc);
            if (C.act == CHAIN_SWISH) return E.template store<DST, CHAIN_SWISH, S>(acc);
        }
        if (C.act == CHAIN_RELU) E.template store<DST, CHAIN_RELU, S>(acc);
        else E.template store<DST, CHAIN_NONE, S>(acc);
    };
    if constexpr (BOTH) {
        if (C.staged) store(std::true_type {});
        else store(std::false_type {});
    } else {
        store(std::integral_constant<bool, FULL> {});
    }
    }
}

template <class Mma, int DST>
int chain_go(chain_more_t &C, unsigned batch, hipStream_t stream, const char *who) {
    constexpr int smem_bytes = line_loader_t<Mma>::LDS_BYTES + CT_BYTES;
    C.tiles_m = (int)((C.M + BM - 1) / BM);
    C.tiles_n = (int)((C.N + Mma::G::BN - 1) / Mma::G::BN);
    const dim3 grid((unsigned)(C.tiles_m * C.tiles_n), 1, DST == CHAIN_PART ? batch * C.split : batch);
    if (const int st = ensure_dynamic_lds((const void *)chain_gemm_kernel<Mma, DST>, smem_bytes, who)) return st;
    hipLaunchKernelGGL((chain_gemm_kernel<Mma, DST>), grid, dim3(Mma::G::NT), smem_bytes, stream, static_cast<const chain_arg_t<DST> &>(C));
    return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
}
// The chain for four consecutive columns of one row, a thread at a time: what chain_part_t::store does with a tile.
// load: its operands, ahead of the sums; m and n are inside dst.
template <int DST>
struct chain_quad_t {
    float ssc, w[4], bias[4];
    v2u_cell_t y;
    __device__ __forceinline__ void load(const chain_t &C, long b, long m, long n) {
        ssc = C.ssc.dt != MI355_DT_UNDEF ? chain_load(C.ssc, b * C.ssc.bs + (C.ssc.per ? m : 0)) : 1.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const long ne = min(n + e, C.N - 1);
            w[e] = C.wsc.dt != MI355_DT_UNDEF ? chain_load(C.wsc, b * C.wsc.bs + (C.wsc.per ? ne : 0)) : 1.f;
            bias[e] = C.bias.dt != MI355_DT_UNDEF ? chain_load(C.bias, b * C.bias.bs + ne) : 0.f;
        }
        if (C.staged) y = *(const v2u_cell_t *)(C.st + b * C.st_bs + m * C.st_pitch + n * 2); // (columns in whole chunks of eight)
    }
    __device__ __forceinline__ void finish(const chain_t &C, long b, long m, long n, float (&x)[4]) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float f = x[e];
            f *= ssc;
            f *= w[e];
            if (C.bias.dt != MI355_DT_UNDEF) f += bias[e];
            if (C.act == CHAIN_RELU) f = DST == CHAIN_I8 ? fmaxf(f, 0.f) : f > 0 ? f : f * 0.f;
            else if (C.act == CHAIN_GELU) f = gelu_tanh_fast(f);
            else if (C.act == CHAIN_SWISH) f = f * logistic_fast(C.alpha * f);
            x[e] = f;
        }
        if (C.staged) {
            const float v[4] = {u2f(y.x << 16), u2f(y.x & 0xffff0000u), u2f(y.y << 16), u2f(y.y & 0xffff0000u)};
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = C.staged == 1 ? x[e] + v[e] : x[e] * v[e];
        }
        constexpr int SHIFT = DST == CHAIN_I8 ? 0 : DST == CHAIN_F32 ? 2 : 1;
        char *to = C.dst + b * C.dst_bs + m * C.dst_pitch + (n << SHIFT);
        const int left = C.N - n < 4 ? (int)(C.N - n) : 4;
        if constexpr (DST == CHAIN_I8) {
            if (C.ds_mode) {
                const float ds = chain_load(chain_vec_t {C.dsc, C.dsc_dt, 0, 0}, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = C.ds_mode == 2 ? x[e] * (1.f / ds) : x[e] / ds;
            }
            const unsigned word = pack4_i8(x, C.lo, C.hi);
            if (left == 4) *(unsigned *)to = word;
            else
                for (int e = 0; e < left; ++e) to[e] = (char)(word >> (8 * e));
        } else if constexpr (DST == CHAIN_F32) {
            if (left == 4) *(v4f *)to = v4f {x[0], x[1], x[2], x[3]};
            else
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (e < left) ((float *)to)[e] = x[e];
        } else {
            v2u_cell_t q;
            if constexpr (DST == CHAIN_F16) {
                unsigned h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = __builtin_bit_cast(uint16_t, (_Float16)x[e]);
                q = v2u_cell_t {h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
            } else {
                bool special = false;
#pragma unroll
                for (int e = 0; e < 4; ++e) special |= __builtin_amdgcn_classf(x[e], 0x93); // NaN or subnormal
                q = chain_bf16(x, __builtin_amdgcn_ballot_w64(special) != 0);
            }
            if (left == 4) *(v2u_cell_t *)to = q;
            else
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    if (e < left) ((uint16_t *)to)[e] = (uint16_t)(q[e / 2] >> (16 * (e % 2)));
        }
    }
};

// K in parts (C.split of them), then their sums and the epilogue
template <class Mma>
int chain_go_parts(int dst_dt, chain_more_t &C, unsigned batch, hipStream_t stream, const char *who) {
    if (const int st = chain_go<Mma, CHAIN_PART>(C, batch, stream, who)) return st;
    return chain_launch_sum(Mma::INTEGER, dst_dt, C, batch, Mma::G::BN == 256, stream);
}
} // namespace
#endif

} // namespace mi355
