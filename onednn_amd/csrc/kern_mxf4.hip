// "hip:mfma_mxf4" -- MXFP4 GEMM: f4_e2m1 x f4_e2m1 with e8m0 block scales over
// 32 consecutive K on both operands, f32 accumulation, on the gfx950
// block-scaled matrix instruction v_mfma_scale_f32_16x16x128_f8f6f4.
//
// Semantics: ref_matmul_t with group_k = 32 (src/cpu/matmul/ref_matmul.cpp:
// 168-236; the Intel GPU reference kernel src/gpu/intel/matmul/ref.cl:200-262
// is the in-tree implementation that runs it):
//   for each block g of 32 k:  acc = sum_j src*wei  (exact in f32)
//                              acc *= 2^(ss-127); acc *= 2^(ws-127); res += acc
// One MFMA covers 128 k = four blocks; lane l carries row l%16 and block l/16,
// i.e. exactly one MX block and one scale byte per operand per lane.  Only the
// rounding of the cross-block f32 additions can differ from the reference.
//
// Operand bytes are K-contiguous nibble pairs; the order of the two nibbles
// inside a byte is irrelevant as long as both operands agree, because all 32
// elements of a block share one scale.
//
// Two small pre-pass kernels of the launch put both operands' scales into the order that the K loop loads them in
// (mx_pack_scales): a stage's scales of 64 rows are 256 contiguous bytes.  From the plain layouts (src [M][K/32] bytes, a
// row's dword of a stage 256 bytes from the next row's at K = 8192) the same load touched 64 cache lines for 256 useful
// bytes, and the scales made as many requests to the L2 as the tiles themselves.
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {
namespace {

using namespace gemm;
using mx_geo_t = geo_t<8, 256>;
using mx_narrow_t = geo_t<4, 128>;

struct mxf4_extra_t {
    const char *bt;       // weights [N][K/2] bytes
    long ldb, bt_bstride; // bytes
    line_scales_args_t sc;
    int tiles_m, tiles_n;
};

struct mxf4_conv_t {
    typedef int row_t;
    template <class PT>
    __device__ __forceinline__ void per_n(const PT &, long, long, float &, int &, int &) const {}
    __device__ __forceinline__ int row_data(long) const { return 0; }
    __device__ __forceinline__ void quad(const v4i_t &raw, int, unsigned, int, float (&f)[4]) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = __int_as_float(raw[e]);
    }
};

extern __shared__ __attribute__((aligned(128))) char mxf4_smem[];

template <class G>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(G::NW / 4))) mxf4_gemm_kernel(const problem_t P_, const mxf4_extra_t X) {
    using Mma = mxf4_mma_t<G>;
    const auto &P = MI355_KERNARG_PROBLEM();
    char *smem = mxf4_smem;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = G::wm(wave), wn = G::wn(wave);
    const long b = blockIdx.z;
    const tile_pos_t tp = tile_position<G>((int)blockIdx.x, X.tiles_m, X.tiles_n);
    const long m0 = tp.m0, n0 = tp.n0;

    const long lda = P.ss[1] / 2; // bytes per src row
    const char *A = (const char *)P.src + (P.ss[0] ? b * (P.ss[0] / 2) : 0) + m0 * lda;
    const char *Bt = X.bt + b * X.bt_bstride + n0 * X.ldb;

    // the epilogue's per-column operands go into their LDS table behind the first loads
    const unsigned ntab = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem + line_loader_t<Mma>::LDS_BYTES;
    auto fill = [&]() __attribute__((always_inline)) { fill_ntab<G::NT>(P, mxf4_conv_t {}, ntab, b, n0); };

    v4f acc[Mma::ROWS][Mma::COLS];
#pragma unroll
    for (int i = 0; i < Mma::ROWS; ++i)
#pragma unroll
        for (int j = 0; j < Mma::COLS; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    main_loop_lines<Mma>(acc, smem, A, Bt, lda, X.ldb, P.M - m0, P.N - n0, P.K / 2, X.sc.tile(b, m0, n0), fill);

    store_quadrant<layout16_t, G::WCOLS>(P, smem, ntab, acc, b, m0 + wm * 128, n0 + wn * G::WCOLS, wn * G::WCOLS,
            mxf4_conv_t {});
}

// in: [R][C] nibbles, C contiguous (two per byte)  ->  out: [C][R] nibbles
__global__ void __launch_bounds__(256) transpose_nibbles_kernel(const uint8_t *in, long R, long C,
        long in_bstride, uint8_t *out, long out_bstride) {
    in += blockIdx.z * in_bstride;
    out += blockIdx.z * out_bstride;
    // one thread per output byte: column c, rows 2r and 2r+1
    const long total = C * (R / 2);
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
            i += (long)gridDim.x * blockDim.x) {
        const long c = i / (R / 2), r2 = i % (R / 2);
        const uint8_t b0 = in[((2 * r2) * C + c) >> 1], b1 = in[((2 * r2 + 1) * C + c) >> 1];
        const uint8_t lo = (c & 1) ? (b0 >> 4) : (b0 & 0xf), hi = (c & 1) ? (b1 >> 4) : (b1 & 0xf);
        out[c * (R / 2) + r2] = (uint8_t)(lo | (hi << 4));
    }
}

// e8m0 scales of `rows` rows x KB blocks of 32 k, element (r, kb) at in[r * rs + kb * ks], into the order the tile
// kernel loads: per stage of 128 k (four blocks) and group of 64 rows 64 dwords, dword 4 r + q = the bytes of block q
// of rows r, 16 + r, 32 + r, 48 + r of the group; groups padded to whole tiles of 256 rows (rows beyond the last
// repeat it).  out[set][group][64] dwords; blocks beyond KB have the scale 1.
// Rows contiguous in the input (weights scales [K/32][N], rs = 1): a thread per dword.
__global__ void __launch_bounds__(256) mx_scales_rows_kernel(const uint8_t *in, long rows, long prows, long KB, long ks,
        long in_bstride, uint32_t *out, long out_bstride) {
    in += blockIdx.z * in_bstride;
    out += blockIdx.z * out_bstride;
    const long nst = (KB + 3) / 4, total = prows * nst;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long st = i / prows, w = i % prows, grp = w / 64;
        const int cell = (int)(w % 64), r = cell >> 2, q = cell & 3;
        const long blk = 4 * st + q;
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            long row = grp * 64 + 16 * e + r;
            row = row < rows ? row : rows - 1;
            v |= (blk < KB ? (uint32_t)in[blk * ks + row] : 127u) << (8 * e);
        }
        out[i] = v;
    }
}
// Blocks contiguous in the input (src scales [M][K/32], ks = 1): a workgroup moves 64 rows x 16 stages through LDS,
// 64 contiguous bytes of a row in, 256 contiguous bytes of a stage and group out.
__global__ void __launch_bounds__(256) mx_scales_blocks_kernel(const uint8_t *in, long rows, long prows, long KB, long rs,
        long in_bstride, uint32_t *out, long out_bstride) {
    __shared__ uint32_t tile[16][65]; // [stage][row]: the row's four block bytes of the stage
    in += blockIdx.z * in_bstride;
    out += blockIdx.z * out_bstride;
    const long grp = blockIdx.x, r0 = grp * 64, q0 = (long)blockIdx.y * 16, nq = (KB + 3) / 4;
    const int t = threadIdx.x;
    const bool aligned = ((uintptr_t)in & 3) == 0 && (rs & 3) == 0 && (KB & 3) == 0;
    {
        const int r = t >> 2, c = t & 3; // row, group of four stages
        const long row = r0 + r < rows ? r0 + r : rows - 1;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const long q = q0 + 4 * c + e;
            const uint8_t *p = in + row * rs + 4 * q;
            uint32_t v = 0u;
            if (q < nq) {
                if (aligned) v = *(const uint32_t *)p; // (KB = rs is whole dwords)
                else
                    for (int x = 3; x >= 0; --x) v = (v << 8) | (4 * q + x < KB ? (uint32_t)p[x] : 127u);
            }
            tile[4 * c + e][r] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int st = (t >> 6) + 4 * e, cell = t & 63, r = cell >> 2, q = cell & 3;
        if (q0 + st < nq) {
            uint32_t v = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) v |= ((tile[st][16 * k + r] >> (8 * q)) & 0xffu) << (8 * k);
            out[(q0 + st) * prows + grp * 64 + cell] = v;
        }
    }
}

struct mxf4_plan_t {
    bool need_transpose;
    size_t off_bt, off_sb, off_sa, off_parts, total;
    chain_split_t split; // of K, where the scratch has room for the parts
    bool small;          // 32 x 32 tiles
    long Bw, Bsb, Bsa;
    long pm, pn; // M, N rounded up to whole tiles
    long nst;
};

// (an f16 dst has a chain on the small tiles only)
bool mxf4_chain(const problem_t &P, bool small, chain_t &C) {
    return chain_from_mx(P, true, false, C)
            && (P.dst_dt == MI355_DT_BF16 || P.dst_dt == MI355_DT_F32 || (small && P.dst_dt == MI355_DT_F16));
}
constexpr long MXF4_STEP_NS = 800; // of a 256 x 128 tile (chain_split)

mxf4_plan_t make_plan(const mi355_matmul_desc_t &d, bool parts) {
    mxf4_plan_t p {};
    p.Bw = d.wei_stride[0] ? d.batch : 1;
    p.Bsb = (d.wei_scale.mask & 1) ? p.Bw : 1;
    p.need_transpose = !(d.wei_stride[1] == 1);
    size_t off = 0;
    p.off_bt = off;
    if (p.need_transpose) off += align_up((size_t)p.Bw * d.N * d.K / 2, 256);
    // the scales in the tile kernel's order, rows padded to whole tiles
    p.pn = (d.N + 255) / 256 * 256;
    p.pm = (d.M + 255) / 256 * 256;
    p.off_sb = off;
    p.nst = (d.K + 127) / 128; // stages, one scale dword per row and stage
    off += align_up((size_t)p.Bsb * p.pn * p.nst * 4, 256);
    p.Bsa = ((d.src_scale.mask & 1) && d.src_stride[0]) ? d.batch : 1;
    p.off_sa = off;
    off += align_up((size_t)p.Bsa * p.pm * p.nst * 4, 256);
    p.off_parts = off;
    p.split = chain_split_t {1, 0};
    problem_t P;
    chain_t C;
    const int force = tuning(TUNE_F8_TILES);
    if (force != TUNE_WIDE && (problem_of_desc(d, P), mxf4_chain(P, true, C))) {
        const bool fits = small_tiles_fit(d.M, d.N, d.K / 2, 4);
        if (parts && !(fits && force == TUNE_SMALL) && P.dst_dt != MI355_DT_F16) p.split = chain_split(d.batch, d.M, d.N, d.K / 2, false, MXF4_STEP_NS);
        p.small = fits
                && (force == TUNE_SMALL
                        || (force == TUNE_AUTO && small_tiles_float(d.batch, d.M, d.N, d.K / 2, p.split, MXF4_STEP_NS, C, 4)));
        if (p.small) p.split = chain_split_t {1, 0};
    }
    off += chain_parts_bytes(d.batch, d.M, d.N, false, p.split.split);
    p.total = off;
    return p;
}

} // namespace

// Packs the e8m0 scales of both operands (src [M][K/32], weights [K/32][N], Bsa / Bsb batches of them) into sa / sb:
// sets of four blocks, (K + 127) / 128 of them, of M / N rounded up to 256 rows, a dword each.
int mx_pack_scales(const mi355_matmul_desc_t &d, const problem_t &P, long Bsa, long Bsb, char *sa, char *sb,
        gemm::line_scales_args_t &sc, hipStream_t stream) {
    const long kb = d.K / 32, sets = (d.K + 127) / 128, pm = (d.M + 255) / 256 * 256, pn = (d.N + 255) / 256 * 256;
    long blocks = (pn * sets + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(mx_scales_rows_kernel, dim3((unsigned)blocks, 1, (unsigned)Bsb), dim3(256), 0, stream,
            (const uint8_t *)P.wei_scale.p, d.N, pn, kb, d.N, kb * d.N, (uint32_t *)sb, pn * sets);
    hipLaunchKernelGGL(mx_scales_blocks_kernel, dim3((unsigned)(pm / 64), (unsigned)((sets + 15) / 16), (unsigned)Bsa),
            dim3(256), 0, stream, (const uint8_t *)P.src_scale.p, d.M, pm, kb, kb, d.M * kb, (uint32_t *)sa, pm * sets);
    sc.a = sa;
    sc.b = sb;
    sc.a_bs = Bsa > 1 ? pm * sets * 4 : 0;
    sc.b_bs = Bsb > 1 ? pn * sets * 4 : 0;
    sc.a_pitch = pm * 4;
    sc.b_pitch = pn * 4;
    sc.sets = (int)sets;
    return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
}

int mxf4_supported(const mi355_matmul_desc_t &d) {
    if (d.src_dt != MI355_DT_F4_E2M1 || d.wei_dt != MI355_DT_F4_E2M1) return MI355_UNIMPLEMENTED;
    if (dt_bits(d.dst_dt) < 8 && !tile_nibble_dst_ok(d)) return MI355_UNIMPLEMENTED;
    // whole MX blocks
    if (d.K < 128 || d.K % 32 != 0) return MI355_UNIMPLEMENTED;
    if (d.src_stride[2] != 1 || d.src_stride[1] % 32 != 0 || d.src_stride[0] % 32 != 0)
        return MI355_UNIMPLEMENTED;
    const bool k_major = d.wei_stride[1] == 1 && d.wei_stride[2] % 32 == 0 && d.wei_stride[0] % 32 == 0;
    const bool n_major = d.wei_stride[2] == 1 && d.wei_stride[1] == d.N && d.N % 2 == 0
            && (d.wei_stride[0] == 0 || d.wei_stride[0] == d.K * d.N);
    if (!k_major && !n_major) return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.src_zp) || !quant_absent(d.wei_zp) || !quant_absent(d.src_pr))
        return MI355_UNIMPLEMENTED;
    // MX scales on both operands: e8m0, one per 32 consecutive k
    const mi355_quant_t &ss = d.src_scale, &ws = d.wei_scale;
    if (ss.dt != MI355_DT_E8M0 || (ss.mask & 6) != 6 || ss.group[0] != 1 || ss.group[1] != 32)
        return MI355_UNIMPLEMENTED;
    if (ws.dt != MI355_DT_E8M0 || (ws.mask & 6) != 6 || ws.group[0] != 32 || ws.group[1] != 1)
        return MI355_UNIMPLEMENTED;
    if (d.batch > 65535) return MI355_UNIMPLEMENTED;
    return MI355_SUCCESS;
}

size_t mxf4_scratch_bytes(const mi355_matmul_desc_t &d, bool parts, size_t *fixed) {
    const mxf4_plan_t p = make_plan(d, parts);
    *fixed = p.off_parts;
    return p.total;
}

int mxf4_launch(const mi355_matmul_desc_t &d, const problem_t &P, const scratch_t &S, hipStream_t stream) {
    const mxf4_plan_t plan = make_plan(d, S.split);
    void *const scratch = S.p;
    if (!scratch) {
        set_error("mfma_mxf4: %zu bytes of scratch required", plan.total);
        return MI355_INVALID_ARGUMENTS;
    }
    char *sc = (char *)scratch;
    mxf4_extra_t X {};
    if (plan.need_transpose) {
        const long total = d.N * (d.K / 2);
        long blocks = (total + 255) / 256;
        if (blocks > 65535) blocks = 65535;
        hipLaunchKernelGGL(transpose_nibbles_kernel, dim3((unsigned)blocks, 1, (unsigned)plan.Bw),
                dim3(256), 0, stream, (const uint8_t *)P.wei, d.K, d.N, d.wei_stride[0] / 2,
                (uint8_t *)(sc + plan.off_bt), d.N * d.K / 2);
        X.bt = sc + plan.off_bt;
        X.ldb = d.K / 2;
        X.bt_bstride = plan.Bw > 1 ? d.N * d.K / 2 : 0;
    } else {
        X.bt = (const char *)P.wei;
        X.ldb = d.wei_stride[2] / 2;
        X.bt_bstride = d.wei_stride[0] / 2;
    }
    // (MI355_F8_TILES keeps one geometry here as well)
    const int force = tuning(TUNE_F8_TILES);
    chain_more_t C {};
    const bool small = plan.small && mxf4_chain(P, true, C), chain = small || mxf4_chain(P, false, C);
    if (!small)
        if (const int st = mx_pack_scales(d, P, plan.Bsa, plan.Bsb, sc + plan.off_sa, sc + plan.off_sb, X.sc, stream)) return st;
    const bool narrow = force == TUNE_NARROW || (line_tiles_narrow(d.batch, d.M, d.N, d.K / 2, chain) && force != TUNE_WIDE);
    if (chain) {
        C.a = (const char *)P.src; C.lda = P.ss[1] / 2; C.a_bs = P.ss[0] / 2;
        C.bt = X.bt; C.ldb = X.ldb; C.b_bs = X.bt_bstride;
        C.kbytes = P.K / 2;
        C.sc = X.sc;
        C.parts = S.parts ? (char *)S.parts : sc + plan.off_parts;
        C.split = plan.split.split;
        C.part_steps = plan.split.part_steps;
        if (small) {
            C.sa = (const uint8_t *)P.src_scale.p; C.sa_bs = plan.Bsa > 1 ? d.M * (d.K / 32) : 0;
            C.sb = (const uint8_t *)P.wei_scale.p; C.sb_bs = plan.Bsb > 1 ? d.N * (d.K / 32) : 0;
            return chain_launch_small(CHAIN_SMALL_MXF4, P.dst_dt, C, (unsigned)d.batch, stream);
        }
        const int st = chain_launch_mx(true, P.dst_dt, C, (unsigned)d.batch, !narrow, stream);
        if (st != MI355_UNIMPLEMENTED) return st;
    }
    if (general_refused("mfma_mxf4")) return MI355_UNIMPLEMENTED;
    X.tiles_m = (int)((d.M + BM - 1) / BM);
    auto go = [&](auto geo) -> int {
        using G = decltype(geo);
        constexpr int smem_bytes = line_loader_t<mxf4_mma_t<G>>::LDS_BYTES + NTAB_BYTES;
        X.tiles_n = (int)((d.N + G::BN - 1) / G::BN);
        const dim3 grid((unsigned)(X.tiles_m * X.tiles_n), 1, (unsigned)d.batch);
        const auto kern = mxf4_gemm_kernel<G>;
        if (const int st = ensure_dynamic_lds((const void *)kern, smem_bytes, "mfma_mxf4")) return st;
        hipLaunchKernelGGL(kern, grid, dim3(G::NT), smem_bytes, stream, P, X);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    // The general epilogue on both tiles: by rounds like the chains, and the narrow one also where one column of them
    // holds N (64 x 4096 x 1024, f16 dst: 25.4 us wide, 21.8 narrow; 300 x 100 x 2048, bf16: 50.6 and 44.5; but 4096 x 4096 x
    // 256, two rounds of narrow tiles: 27.2 and 39.3).
    return narrow || (d.N <= mx_narrow_t::BN && force != TUNE_WIDE) ? go(mx_narrow_t {}) : go(mx_geo_t {});
}

} // namespace mi355
