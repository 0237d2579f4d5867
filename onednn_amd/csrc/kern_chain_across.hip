// hip:mfma_h16 on the chain kernels (chain_gemm.hpp) with operands that are contiguous across K: backward by data (the
// weights) and by weights (both) of a linear layer read them where they lie.
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {

int chain_launch_h16_across(bool bf16, int dst_dt, int across, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
    using narrow_t = geo_t<4, 128>;
    using wide_t = geo_t<8, 256>;
    auto go = [&](auto b16, auto dst) -> int {
        constexpr bool B = decltype(b16)::value;
        constexpr int D = decltype(dst)::value;
        if (across == 2) return chain_go<h16_across_mma_t<B, wide_t, 2>, D>(C, batch, stream, "mfma_h16");
        return wide ? chain_go<h16_across_mma_t<B, wide_t, 1>, D>(C, batch, stream, "mfma_h16")
                    : chain_go<h16_across_mma_t<B, narrow_t, 1>, D>(C, batch, stream, "mfma_h16");
    };
    if (C.split > 1) {
        auto parts = [&](auto b16) -> int {
            constexpr bool B = decltype(b16)::value;
            return across == 2 ? chain_go_parts<h16_across_mma_t<B, wide_t, 2>>(dst_dt, C, batch, stream, "mfma_h16")
                               : chain_go_parts<h16_across_mma_t<B, narrow_t, 1>>(dst_dt, C, batch, stream, "mfma_h16");
        };
        return bf16 ? parts(std::true_type {}) : parts(std::false_type {});
    }
    constexpr std::integral_constant<int, CHAIN_F32> f32 {};
    if (bf16 && dst_dt == MI355_DT_BF16) return go(std::true_type {}, std::integral_constant<int, CHAIN_BF16> {});
    if (bf16 && dst_dt == MI355_DT_F32) return go(std::true_type {}, f32);
    if (!bf16 && dst_dt == MI355_DT_F16) return go(std::false_type {}, std::integral_constant<int, CHAIN_F16> {});
    if (!bf16 && dst_dt == MI355_DT_F32) return go(std::false_type {}, f32);
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
