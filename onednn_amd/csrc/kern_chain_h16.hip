// hip:mfma_h16 on the chain kernels (chain_gemm.hpp), and which problems those take.
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {

bool chain_form(const problem_t &P, bool scaled, bool full, chain_t &C) {
    const int db = dt_bits(P.dst_dt);
    if (P.dst_dt != MI355_DT_BF16 && P.dst_dt != MI355_DT_F16 && P.dst_dt != MI355_DT_F32 && !is_int8_dt(P.dst_dt)) return false;
    if (P.rnd_flags || P.dst_dynamic || P.dst_zp.dt != MI355_DT_UNDEF || P.ds[2] != 1) return false;
    C = chain_t {};
    // rows of whole 16-byte pieces; 8-bit ones may start at any dword (they leave in dwords then)
    const long esz = db / 8, align = db == 8 ? 4 : 16;
    C.dst = (char *)P.dst;
    C.dst_pitch = P.ds[1] * esz;
    C.dst_bs = P.B > 1 ? P.ds[0] * esz : 0;
    if ((C.dst_pitch | C.dst_bs) & (align - 1)) return false;
    C.M = P.M;
    C.N = P.N;
    auto readable = [](int dt) { return dt == MI355_DT_F32 || dt == MI355_DT_BF16 || dt == MI355_DT_F16; };
    if (scaled) {
        if (P.src_scale.dt != MI355_DT_UNDEF) {
            if (!readable(P.src_scale.dt) || (P.src_scale.mask & 4)) return false;
            C.ssc = {P.src_scale.p, P.src_scale.dt, (P.src_scale.mask & 2) != 0, 0};
            if ((P.src_scale.mask & 1) && P.ss[0]) C.ssc.bs = C.ssc.per ? P.M : 1;
        }
        if (P.wei_scale.dt != MI355_DT_UNDEF) {
            if (!readable(P.wei_scale.dt) || (P.wei_scale.mask & 2)) return false;
            C.wsc = {P.wei_scale.p, P.wei_scale.dt, (P.wei_scale.mask & 4) != 0, 0};
            if ((P.wei_scale.mask & 1) && P.ws[0]) C.wsc.bs = C.wsc.per ? P.N : 1;
        }
    } else if (P.src_scale.dt != MI355_DT_UNDEF || P.wei_scale.dt != MI355_DT_UNDEF) {
        return false;
    }
    if (P.bias_dt != MI355_DT_UNDEF) {
        if (!readable(P.bias_dt) || P.bs[1] != 0 || P.bs[2] != 1) return false;
        C.bias = {P.bias, P.bias_dt, 1, P.bs[0]};
    }
    if (P.dst_scale.dt != MI355_DT_UNDEF) {
        if (db != 8 || !readable(P.dst_scale.dt) || P.dst_scale.mask != 0) return false;
        C.dsc = P.dst_scale.p;
        C.dsc_dt = P.dst_scale.dt;
        C.ds_mode = P.dst_scale_mode == MI355_DST_SCALE_RECIPROCAL ? 2 : 1;
    }
    C.lo = P.dst_dt == MI355_DT_S8 ? -128 : 0;
    C.hi = P.dst_dt == MI355_DT_S8 ? 127 : 255;
    // [activation] [bf16 tensor]
    const bool all = full && db == 16;
    int at = 0;
    if (at < P.n_po && P.po[at].kind == MI355_PO_ELTWISE && P.po[at].scale == 1.f) {
        const auto &e = P.po[at];
        if (e.alg == MI355_ELTWISE_RELU && e.alpha == 0.f) C.act = CHAIN_RELU;
        else if (all && e.alg == MI355_ELTWISE_GELU_TANH) C.act = CHAIN_GELU;
        else if (all && e.alg == MI355_ELTWISE_SWISH) C.act = CHAIN_SWISH;
        else return false;
        C.alpha = e.alpha;
        ++at;
    }
    if (at < P.n_po && P.po[at].kind == MI355_PO_BINARY) {
        const auto &y = P.po[at];
        if (!all || y.dt != MI355_DT_BF16 || (y.alg != MI355_BINARY_ADD && y.alg != MI355_BINARY_MUL)) return false;
        // whole 16-byte pieces of every row, with rows of their own (the loads are 32-bit offsets from a tile's first row)
        if (y.s1 == 0 || y.s2 != 1 || ((uintptr_t)y.p & 15) || (P.B > 1 && y.s0 % 8) || y.s1 % 8 || P.N % 8 || y.s1 < 0 || y.s1 >= (1L << 22)) return false;
        C.staged = y.alg == MI355_BINARY_ADD ? 1 : 2;
        C.st = (const char *)y.p;
        C.st_pitch = y.s1 * 2;
        C.st_bs = y.s0 * 2;
        ++at;
    }
    return at == P.n_po;
}

bool chain_from(const problem_t &P, bool scaled, bool full, chain_t &C) {
    return chain_form(P, scaled, full, C) && chain_dst_aligned(C, P.dst_dt);
}

bool chain_from_mx(const problem_t &P, bool mx, bool full, chain_t &C) {
    if (!mx) return chain_from(P, true, full, C);
    problem_t Q = P;
    Q.src_scale.dt = Q.wei_scale.dt = MI355_DT_UNDEF;
    return chain_from(Q, false, full, C);
}

int chain_launch_h16(bool bf16, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
    using narrow_t = geo_t<4, 128>;
    using wide_t = geo_t<8, 256>;
    auto go = [&](auto b16, auto dst) -> int {
        constexpr bool B = decltype(b16)::value;
        constexpr int D = decltype(dst)::value;
        return wide ? chain_go<h16x16_mma_t<B, wide_t>, D>(C, batch, stream, "mfma_h16")
                    : chain_go<h16x16_mma_t<B, narrow_t>, D>(C, batch, stream, "mfma_h16");
    };
    auto go_mixed = [&](auto b16, auto dst) -> int {
        constexpr bool B = decltype(b16)::value;
        constexpr int D = decltype(dst)::value;
        return wide ? chain_go<h16_mixed_mma_t<B, wide_t>, D>(C, batch, stream, "mfma_h16")
                    : chain_go<h16_mixed_mma_t<B, narrow_t>, D>(C, batch, stream, "mfma_h16");
    };
    if (C.split > 1)
        return bf16 ? chain_go_parts<h16x16_mma_t<true, narrow_t>>(dst_dt, C, batch, stream, "mfma_h16")
                    : chain_go_parts<h16x16_mma_t<false, narrow_t>>(dst_dt, C, batch, stream, "mfma_h16");
    constexpr std::integral_constant<int, CHAIN_F32> f32 {};
    constexpr std::integral_constant<int, CHAIN_BF16> b {};
    constexpr std::integral_constant<int, CHAIN_F16> h {};
    if (bf16 && dst_dt == MI355_DT_BF16) return go(std::true_type {}, b);
    if (bf16 && dst_dt == MI355_DT_F16) return go_mixed(std::true_type {}, h);
    if (bf16 && dst_dt == MI355_DT_F32) return go(std::true_type {}, f32);
    if (!bf16 && dst_dt == MI355_DT_BF16) return go_mixed(std::false_type {}, b);
    if (!bf16 && dst_dt == MI355_DT_F16) return go(std::false_type {}, h);
    if (!bf16 && dst_dt == MI355_DT_F32) return go(std::false_type {}, f32);
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
