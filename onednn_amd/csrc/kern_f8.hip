// "hip:mfma_f8" -- LDS-tiled fp8 GEMM (OCP e4m3 / e5m2 operands, f32
// accumulation) on the gfx950 matrix cores, v_mfma_f32_16x16x128_f8f6f4, with
// the reference's epilogue fused in.
//
// Semantics: ref_matmul_t (src/cpu/matmul/ref_matmul.cpp:168-331) for f8 src
// and weights with per-tensor / per-row src scales and per-tensor / per-n
// weights scales.  The reference scales every product before summing
// (its "group" is a single k when no K groups exist); this kernel sums the
// exact e4m3 x e4m3 products in f32 on the matrix cores and applies
//   acc * src_scale * wei_scale
// once, which differs only in rounding and is covered by the f32/bf16
// comparison thresholds.
#include <algorithm>
#include <cstring>
#include "f8_family.hpp"
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {
namespace {

// MXFP8: ref_matmul_t with group_k = 32 -- acc = sum of a block's 32 products, acc *= 2^(ss-127), acc *= 2^(ws-127),
// res += acc (src/cpu/matmul/ref_matmul.cpp:168-236) -- on the scaled instruction (mxf8_mma_t, line_policies.hpp).  A
// pre-pass of the launch packs the scales (mx_pack_scales, kern_mxf4.hip).
struct f8_plan_t {
    bool need_transpose, mx;
    size_t off_sa, off_sb, off_parts, total;
    chain_split_t split; // of K, where the scratch has room for the parts
    bool small;          // 32 x 32 tiles
    long Bw, Bsa, Bsb;
    long sets, pm, pn; // MX: sets of four blocks of K; M, N rounded up to whole tiles
};

// MX: e8m0 scales per 32 consecutive k on both operands
bool f8_is_mx(const mi355_matmul_desc_t &d) {
    const mi355_quant_t &ss = d.src_scale, &ws = d.wei_scale;
    return ss.dt == MI355_DT_E8M0 && (ss.mask & 6) == 6 && ss.group[0] == 1 && ss.group[1] == 32
            && ws.dt == MI355_DT_E8M0 && (ws.mask & 6) == 6 && ws.group[0] == 32 && ws.group[1] == 1;
}

bool is_e4m3_pair(const mi355_matmul_desc_t &d) { return d.src_dt == MI355_DT_F8_E4M3 && d.wei_dt == MI355_DT_F8_E4M3; }
// (an f16 dst has a chain on the small tiles only)
bool f8_chain(const problem_t &P, bool mx, bool small, chain_t &C) {
    return chain_from_mx(P, mx, true, C)
            && (P.dst_dt == MI355_DT_BF16 || P.dst_dt == MI355_DT_F32 || (small && P.dst_dt == MI355_DT_F16));
}
constexpr long F8_STEP_NS = 700; // of a 256 x 128 tile (chain_split)

f8_plan_t make_plan(const mi355_matmul_desc_t &d, bool parts) {
    f8_plan_t p {};
    p.Bw = d.wei_stride[0] ? d.batch : 1;
    p.need_transpose = !(d.wei_stride[1] == 1);
    p.mx = f8_is_mx(d);
    p.Bsb = (d.wei_scale.mask & 1) ? p.Bw : 1;
    p.Bsa = ((d.src_scale.mask & 1) && d.src_stride[0]) ? d.batch : 1;
    size_t off = p.need_transpose ? align_up((size_t)p.Bw * d.N * d.K, 256) : 0;
    if (p.mx) { // the packed scales of both operands
        p.sets = (d.K + 127) / 128;
        p.pm = (d.M + 255) / 256 * 256;
        p.pn = (d.N + 255) / 256 * 256;
        // a dword per row and set fits into 256 bytes per 64 bytes of K and 128 rows (one block of them to spare) or 64
        // columns but for an odd number of 64 bytes; the size has always been the latter
        const long stages = (d.K + 63) / 64;
        p.off_sa = off;
        off += align_up((size_t)p.Bsa * std::max(p.pm * p.sets * 4, ((d.M + 127) / 128 + 1) * stages * 256), 256);
        p.off_sb = off;
        off += align_up((size_t)p.Bsb * std::max(p.pn * p.sets * 4, p.pn * 4 * stages), 256);
    }
    p.off_parts = off;
    p.split = chain_split_t {1, 0};
    problem_t P;
    chain_t C;
    const int force = tuning(TUNE_F8_TILES);
    if (is_e4m3_pair(d) && force != TUNE_WIDE && (problem_of_desc(d, P), f8_chain(P, p.mx, true, C))) {
        const bool fits = small_tiles_fit(d.M, d.N, d.K, p.mx ? 8 : 0);
        if (parts && !(fits && force == TUNE_SMALL) && P.dst_dt != MI355_DT_F16) p.split = chain_split(d.batch, d.M, d.N, d.K, false, F8_STEP_NS);
        p.small = fits
                && (force == TUNE_SMALL
                        || (force == TUNE_AUTO && small_tiles_float(d.batch, d.M, d.N, d.K, p.split, F8_STEP_NS, C, p.mx ? 8 : 0)));
        if (p.small) p.split = chain_split_t {1, 0};
    }
    off += chain_parts_bytes(d.batch, d.M, d.N, false, p.split.split);
    p.total = off;
    return p;
}

} // namespace

int f8_supported(const mi355_matmul_desc_t &d) {
    if (!is_f8_dt(d.src_dt) || !is_f8_dt(d.wei_dt)) return MI355_UNIMPLEMENTED;
    if (dt_bits(d.dst_dt) < 8 && !tile_nibble_dst_ok(d)) return MI355_UNIMPLEMENTED;
    // whole 16-byte chunks of K
    if (d.K < 64 || d.K % 16 != 0) return MI355_UNIMPLEMENTED;
    if (d.src_stride[2] != 1 || d.src_stride[1] % 16 != 0 || d.src_stride[0] % 16 != 0)
        return MI355_UNIMPLEMENTED;
    const bool k_major = d.wei_stride[1] == 1 && d.wei_stride[2] % 16 == 0 && d.wei_stride[0] % 16 == 0;
    const bool n_major = d.wei_stride[2] == 1;
    if (!k_major && !n_major) return MI355_UNIMPLEMENTED;
    // no zero points on this path, scales without groups and without a K mask
    if (!quant_absent(d.src_zp) || !quant_absent(d.wei_zp) || !quant_absent(d.src_pr))
        return MI355_UNIMPLEMENTED;
    if (f8_is_mx(d)) {
        // whole blocks of 32 k, static dst quantization
        if (d.K % 32 != 0 || d.dst_scale_dynamic != MI355_DST_DYNAMIC_NONE) return MI355_UNIMPLEMENTED;
        if (d.batch > 65535) return MI355_UNIMPLEMENTED;
        return MI355_SUCCESS;
    }
    if (!quant_absent(d.src_scale)
            && ((d.src_scale.mask & 4) || d.src_scale.group[0] > 1 || d.src_scale.group[1] > 1))
        return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.wei_scale)
            && ((d.wei_scale.mask & 2) || d.wei_scale.group[0] > 1 || d.wei_scale.group[1] > 1))
        return MI355_UNIMPLEMENTED;
    if (d.batch > 65535) return MI355_UNIMPLEMENTED;
    return MI355_SUCCESS;
}

size_t f8_scratch_bytes(const mi355_matmul_desc_t &d, bool parts, size_t *fixed) {
    const f8_plan_t p = make_plan(d, parts);
    *fixed = p.off_parts;
    return p.total;
}

int f8_launch(const mi355_matmul_desc_t &d, const problem_t &P, const scratch_t &S, hipStream_t stream) {
    const f8_plan_t plan = make_plan(d, S.split);
    void *const scratch = S.p;
    if (plan.total > 0 && !scratch) {
        set_error("mfma_f8: %zu bytes of scratch required", plan.total);
        return MI355_INVALID_ARGUMENTS;
    }
    f8_extra_t X {};
    if (plan.need_transpose) {
        transpose_bytes(P.wei, d.K, d.N, d.wei_stride[1], d.wei_stride[0], scratch, d.K, d.N * d.K,
                plan.Bw, stream);
        X.bt = (const char *)scratch;
        X.ldb = d.K;
        X.bt_bstride = plan.Bw > 1 ? d.N * d.K : 0;
    } else {
        X.bt = (const char *)P.wei;
        X.ldb = d.wei_stride[2];
        X.bt_bstride = d.wei_stride[0];
    }
    const int fa = d.src_dt == MI355_DT_F8_E5M2, fb = d.wei_dt == MI355_DT_F8_E5M2;
    chain_more_t C {};
    const bool small = plan.small && f8_chain(P, plan.mx, true, C);
    const bool chain = small || (is_e4m3_pair(d) && f8_chain(P, plan.mx, false, C));
    if (plan.mx && !small) {
        char *sa = (char *)scratch + plan.off_sa, *sb = (char *)scratch + plan.off_sb;
        if (const int st = mx_pack_scales(d, P, plan.Bsa, plan.Bsb, sa, sb, X.sc, stream)) return st;
    }
    // (MI355_F8_TILES: wide / narrow keep one geometry whatever the size: tests, tuning)
    const int force = tuning(TUNE_F8_TILES);
    const bool narrow = force == TUNE_NARROW || (line_tiles_narrow(d.batch, d.M, d.N, d.K, chain) && force != TUNE_WIDE);
    if (chain) {
        C.a = (const char *)P.src; C.lda = P.ss[1]; C.a_bs = P.ss[0];
        C.bt = X.bt; C.ldb = X.ldb; C.b_bs = X.bt_bstride;
        C.kbytes = P.K;
        C.sc = X.sc;
        C.parts = S.parts ? (char *)S.parts : (char *)scratch + plan.off_parts;
        C.split = plan.split.split;
        C.part_steps = plan.split.part_steps;
        if (small) {
            C.sa = (const uint8_t *)P.src_scale.p; C.sa_bs = plan.Bsa > 1 ? d.M * (d.K / 32) : 0;
            C.sb = (const uint8_t *)P.wei_scale.p; C.sb_bs = plan.Bsb > 1 ? d.N * (d.K / 32) : 0;
            return chain_launch_small(plan.mx ? CHAIN_SMALL_MXF8 : CHAIN_SMALL_F8, P.dst_dt, C, (unsigned)d.batch, stream);
        }
        const int st = plan.mx ? chain_launch_mx(false, P.dst_dt, C, (unsigned)d.batch, !narrow, stream)
                               : chain_launch_f8(P.dst_dt, C, (unsigned)d.batch, !narrow, stream);
        if (st != MI355_UNIMPLEMENTED) return st;
    }
    if (general_refused("mfma_f8")) return MI355_UNIMPLEMENTED;
    if (narrow && !plan.mx) return f8_launch_narrow(fa, fb, P, X.bt, X.ldb, X.bt_bstride, (unsigned)d.batch, stream);
    X.tiles_m = (int)((d.M + BM - 1) / BM);
    X.tiles_n = (int)((d.N + f8_geo_t::BN - 1) / f8_geo_t::BN);
    const dim3 grid((unsigned)(X.tiles_m * X.tiles_n), 1, (unsigned)d.batch);
    auto go = [&](auto mma) -> int {
        using Mma = decltype(mma);
        constexpr int smem_bytes = ring_of<Mma>::BYTES + NTAB_BYTES;
        const auto kern = f8_gemm_kernel<Mma>;
        if (const int st = ensure_dynamic_lds((const void *)kern, smem_bytes, "mfma_f8")) return st;
        hipLaunchKernelGGL(kern, grid, dim3(f8_geo_t::NT), smem_bytes, stream, P, X);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    if (plan.mx) {
        if (fa && fb) return go(mxf8_mma_t<1, 1, f8_geo_t> {});
        if (fa) return go(mxf8_mma_t<1, 0, f8_geo_t> {});
        if (fb) return go(mxf8_mma_t<0, 1, f8_geo_t> {});
        return go(mxf8_mma_t<0, 0, f8_geo_t> {});
    }
    if (fa && fb) return go(f8_mma_t<1, 1, f8_geo_t> {});
    if (fa) return go(f8_mma_t<1, 0, f8_geo_t> {});
    if (fb) return go(f8_mma_t<0, 1, f8_geo_t> {});
    return go(f8_mma_t<0, 0, f8_geo_t> {});
}

} // namespace mi355
