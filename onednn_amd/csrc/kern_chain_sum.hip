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
__global__ void __launch_bounds__(256) chain_sum_kernel(const chain_more_t C) {
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
    chain_quad_t<DST> Q;
    Q.load(C, b, m, n);
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

    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (INTEGER) {
            const int a = C.off_s - (C.src_zp ? *C.src_zp : 0);
            x[e] = (float)(sum[e] + (C.colsum ? a * C.colsum[b * C.colsum_bs + min(n + e, C.N - 1)] : 0));
        } else {
            x[e] = sum[e];
        }
    }
    Q.finish(C, b, m, n, x);
}

} // namespace

int chain_launch_sum(bool integer, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
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
