// The sums of a product whose K was split over workgroups (chain_gemm.hpp, CHAIN_PART), and its epilogue.
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {
namespace {

// A thread owns a quad of accumulators, four consecutive columns of a row; a workgroup the 16 rows x 64 columns of one row
// block of a wavefront's part, a quad column a wavefront.  Parts are added in their order, so results do not depend on
// timing.  Bound: the parts' bytes (they were written a moment ago and come from the memory-side cache) and, for small
// problems, the launch.
template <bool INTEGER, int DST, class G>
__global__ void __launch_bounds__(256) chain_sum_kernel(const chain_t C) {
    using V = std::conditional_t<INTEGER, v4i, v4f>;
    const int t = threadIdx.x, lane = t & 63, k = t >> 6;
    const int i = blockIdx.x % 8, wave = blockIdx.x / 8 % G::NW, id = blockIdx.x / (8 * G::NW);
    const long b = blockIdx.z, tiles = (long)C.tiles_m * C.tiles_n;
    const tile_pos_t tp = tile_position<G>(id, C.tiles_m, C.tiles_n);
    const long m = tp.m0 + G::wm(wave) * 128 + 16 * i + (lane & 15);
    const long n = tp.n0 + G::wn(wave) * 64 + 16 * k + 4 * (lane >> 4);
    if (m >= C.M || n >= C.N) return;
    const char *from = C.parts + ((b * C.split * tiles + id) * G::NW + wave) * 32768 + (i * 4 + k) * 1024 + lane * 16;
    const long pitch = tiles * G::NW * 32768;
    const float ssc = C.ssc.dt != MI355_DT_UNDEF ? chain_load(C.ssc, b * C.ssc.bs + (C.ssc.per ? m : 0)) : 1.f;
    float w[4], bias[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const long ne = min(n + e, C.N - 1);
        w[e] = C.wsc.dt != MI355_DT_UNDEF ? chain_load(C.wsc, b * C.wsc.bs + (C.wsc.per ? ne : 0)) : 1.f;
        bias[e] = C.bias.dt != MI355_DT_UNDEF ? chain_load(C.bias, b * C.bias.bs + ne) : 0.f;
    }
    V sum = *(const V *)from;
    int p = 1;
    for (; p + 4 <= C.split; p += 4) {
        V q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = *(const V *)(from + (p + u) * pitch);
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += q[u];
    }
    for (; p < C.split; ++p) sum += *(const V *)(from + p * pitch);

    // the chain, step by step as chain_part_t::store takes it
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float f;
        if constexpr (INTEGER) {
            const int a = C.off_s - (C.src_zp ? *C.src_zp : 0);
            f = (float)(sum[e] + (C.colsum ? a * C.colsum[b * C.colsum_bs + min(n + e, C.N - 1)] : 0));
        } else {
            f = sum[e];
        }
        f *= ssc;
        f *= w[e];
        if (C.bias.dt != MI355_DT_UNDEF) f += bias[e];
        if (C.act == CHAIN_RELU) f = DST == CHAIN_I8 ? fmaxf(f, 0.f) : f > 0 ? f : f * 0.f;
        else if (C.act == CHAIN_GELU) f = gelu_tanh_fast(f);
        else if (C.act == CHAIN_SWISH) f = f * logistic_fast(C.alpha * f);
        x[e] = f;
    }
    if (C.staged) { // (columns in whole chunks of eight)
        const v2u_cell_t q = *(const v2u_cell_t *)(C.st + b * C.st_bs + m * C.st_pitch + n * 2);
        const float y[4] = {u2f(q.x << 16), u2f(q.x & 0xffff0000u), u2f(q.y << 16), u2f(q.y & 0xffff0000u)};
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = C.staged == 1 ? x[e] + y[e] : x[e] * y[e];
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

} // namespace

int chain_launch_sum(bool integer, int dst_dt, chain_t &C, unsigned batch, bool wide, hipStream_t stream) {
    auto go = [&](auto is_int, auto dst, auto geo) -> int {
        using G = decltype(geo);
        hipLaunchKernelGGL((chain_sum_kernel<decltype(is_int)::value, decltype(dst)::value, G>),
                dim3((unsigned)(C.tiles_m * C.tiles_n * G::NW * 8), 1, batch), dim3(256), 0, stream, C);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    auto tile = [&](auto is_int, auto dst) -> int { return wide ? go(is_int, dst, geo_t<8, 256> {}) : go(is_int, dst, geo_t<4, 128> {}); };
    constexpr std::integral_constant<int, CHAIN_BF16> b16 {};
    constexpr std::integral_constant<int, CHAIN_F32> f32 {};
    if (integer) {
        constexpr geo_t<4, 128> narrow {};
        if (is_int8_dt(dst_dt)) return go(std::true_type {}, std::integral_constant<int, CHAIN_I8> {}, narrow);
        if (dst_dt == MI355_DT_BF16) return go(std::true_type {}, b16, narrow);
        if (dst_dt == MI355_DT_F32) return go(std::true_type {}, f32, narrow);
        return MI355_UNIMPLEMENTED;
    }
    if (dst_dt == MI355_DT_BF16) return tile(std::false_type {}, b16);
    if (dst_dt == MI355_DT_F16) return tile(std::false_type {}, std::integral_constant<int, CHAIN_F16> {});
    if (dst_dt == MI355_DT_F32) return tile(std::false_type {}, f32);
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
