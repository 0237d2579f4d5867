// What the fp8 family ("hip:mfma_f8", kern_f8.hip) and the unquantized float family ("hip:mfma_h16", kern_h16.hip)
// share: the general kernel -- any epilogue, from the problem's description -- over an operand policy, and the scale
// handling.
#pragma once
#include <type_traits>

#include "line_loops.hpp"

namespace mi355 {
namespace {

using namespace gemm;
using f8_geo_t = geo_t<8, 256>;
using narrow_geo_t = geo_t<4, 128>;

struct f8_extra_t {
    const char *bt; // weights as [N][K] bytes, K contiguous
    long ldb, bt_bstride;
    int tiles_m, tiles_n;
    line_scales_args_t sc; // block-scaled policies: the e8m0 scales per 32 k of both operands, packed by a pre-pass
};

struct f8_conv_t {
    typedef float row_t;
    float ssc_common;
    const void *ssc_p; // per-row src scales (already offset to this batch) or null
    int ssc_dt;
    bool with_src_sc, with_wei_sc;
    long bw;
    template <class PT>
    __device__ __forceinline__ void per_n(const PT &P, long, long n, float &wsc, int &, int &) const {
        if (with_wei_sc)
            wsc = load_float(P.wei_scale.dt, P.wei_scale.p, quant_off(P.wei_scale, bw, 0, n, P.K, P.N));
    }
    __device__ __forceinline__ float row_data(long m) const {
        return ssc_p ? load_float(ssc_dt, ssc_p, m) : ssc_common;
    }

    __device__ __forceinline__ void quad(const v4i_t &raw, float ssc, unsigned ntab, int col, float (&f)[4]) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = __int_as_float(raw[e]);
        if (with_src_sc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] *= ssc;
        }
        if (with_wei_sc) {
            const v4f_t w = nt4f(ntab, NT_WSC, col);
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] *= w[e];
        }
    }
};

// accumulator tile of a policy: 32 x 32 (sixteen registers) unless it declares TILE16
template <class Mma, class = void>
struct acc_of {
    typedef v16f type;
    typedef layout32_t layout;
    static constexpr int N = 16;
};
template <class Mma>
struct acc_of<Mma, std::enable_if_t<Mma::TILE16>> {
    typedef v4f type;
    typedef layout16_t layout;
    static constexpr int N = 4;
};

// block-scaled policies (MX = true)
template <class Mma, class = void>
struct mx_of : std::false_type {};
template <class Mma>
struct mx_of<Mma, std::enable_if_t<Mma::MX>> : std::true_type {};

// LDS of a policy's K loop, wavefronts per SIMD
template <class Mma, class = void>
struct ring_of {
    static constexpr int BYTES = Mma::G::NSTAGE * Mma::G::STAGE_BYTES;
    static constexpr int WAVES = Mma::G::NW / 4;
};
template <class Mma>
struct ring_of<Mma, std::enable_if_t<reads_lines<Mma>::value>> {
    static constexpr int BYTES = line_loader_t<Mma>::LDS_BYTES;
    static constexpr int WAVES = Mma::G::NW / 4;
};

extern __shared__ __attribute__((aligned(128))) char f8_smem[];

template <class Mma>
__global__ void __launch_bounds__(Mma::G::NT) __attribute__((amdgpu_waves_per_eu(ring_of<Mma>::WAVES))) f8_gemm_kernel(const problem_t P_, const f8_extra_t X) {
    using G = typename Mma::G;
    constexpr int EB = Mma::ELEM_BYTES;
    const auto &P = MI355_KERNARG_PROBLEM();
    char *smem = f8_smem;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = G::wm(wave), wn = G::wn(wave);
    const long b = blockIdx.z;
    const tile_pos_t tp = tile_position<G>((int)blockIdx.x, X.tiles_m, X.tiles_n);
    const long m0 = tp.m0, n0 = tp.n0;

    const long lda = P.ss[1] * EB; // bytes, like X.ldb and X.bt_bstride
    const char *A = (const char *)P.src + (P.ss[0] ? b * P.ss[0] * EB : 0) + m0 * lda;
    const char *Bt = X.bt + b * X.bt_bstride + n0 * X.ldb;

    const long bs = P.ss[0] ? b : 0, bw = P.ws[0] ? b : 0;
    f8_conv_t cv;
    // (block scales are operands of the instruction: nothing of them is left for the epilogue)
    cv.with_src_sc = !mx_of<Mma>::value && P.src_scale.dt != MI355_DT_UNDEF;
    cv.with_wei_sc = !mx_of<Mma>::value && P.wei_scale.dt != MI355_DT_UNDEF;
    cv.ssc_common = 1.f;
    cv.ssc_p = nullptr;
    cv.ssc_dt = mx_of<Mma>::value ? (int)MI355_DT_UNDEF : P.src_scale.dt;
    cv.bw = bw;
    if (cv.with_src_sc) {
        if (P.src_scale.mask & 2)
            cv.ssc_p = (const char *)P.src_scale.p
                    + ((P.src_scale.mask & 1) ? bs * P.M : 0) * (dt_bits(P.src_scale.dt) / 8);
        else
            cv.ssc_common = load_float(P.src_scale.dt, P.src_scale.p, (P.src_scale.mask & 1) ? bs : 0);
    }
    // the epilogue's per-column operands go into their LDS table now: the loads
    // hide behind the pipeline prologue
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;
    const unsigned ntab = lds0 + ring_of<Mma>::BYTES;
    auto fill = [&]() __attribute__((always_inline)) { fill_ntab<G::NT>(P, cv, ntab, b, n0); };
    if constexpr (!reads_lines<Mma>::value) fill();

    typename acc_of<Mma>::type acc[Mma::ROWS][Mma::COLS];
#pragma unroll
    for (int i = 0; i < Mma::ROWS; ++i)
#pragma unroll
        for (int j = 0; j < Mma::COLS; ++j)
#pragma unroll
            for (int r = 0; r < acc_of<Mma>::N; ++r) acc[i][j][r] = 0.f;

    const long kbytes = P.K * EB;
    if constexpr (reads_lines<Mma>::value)
        main_loop_lines<Mma>(acc, smem, A, Bt, lda, X.ldb, P.M - m0, P.N - n0, kbytes, X.sc.tile(b, m0, n0), fill);
    else
        main_loop_two_groups<G::NSTAGE, Mma>(acc, smem, A, Bt, lda, X.ldb, P.M - m0, P.N - n0, (int)(kbytes / BKB));

    store_quadrant<typename acc_of<Mma>::layout, G::WCOLS>(P, smem, ntab, acc, b, m0 + wm * 128, n0 + wn * G::WCOLS,
            wn * G::WCOLS, cv);
}

} // namespace
} // namespace mi355
