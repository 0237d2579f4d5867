// hip:mfma_i8 on the chain kernels (chain_gemm.hpp).
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {

int chain_launch_i8(bool src_u8, int dst_dt, chain_t &C, unsigned batch, bool wide, hipStream_t stream) {
    auto go = [&](auto u8, auto dst) -> int {
        constexpr bool U = decltype(u8)::value;
        constexpr int D = decltype(dst)::value;
        return wide ? chain_go<i8_mma_t<U, false, geo_t<8, 256>>, D>(C, batch, stream, "mfma_i8")
                    : chain_go<i8_mma_t<U, false, geo_t<4, 128>>, D>(C, batch, stream, "mfma_i8");
    };
    auto by_dst = [&](auto u8) -> int {
        if (is_int8_dt(dst_dt)) return go(u8, std::integral_constant<int, CHAIN_I8> {});
        if (dst_dt == MI355_DT_BF16) return go(u8, std::integral_constant<int, CHAIN_BF16> {});
        if (dst_dt == MI355_DT_F32) return go(u8, std::integral_constant<int, CHAIN_F32> {});
        return MI355_UNIMPLEMENTED;
    };
    return src_u8 ? by_dst(std::true_type {}) : by_dst(std::false_type {});
}

} // namespace mi355
