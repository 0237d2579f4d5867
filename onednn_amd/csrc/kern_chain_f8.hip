// hip:mfma_f8, e4m3 x e4m3, on the chain kernels (chain_gemm.hpp).
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {

int chain_launch_f8(int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
    auto go = [&](auto dst) -> int {
        constexpr int D = decltype(dst)::value;
        return wide ? chain_go<f8_mma_t<0, 0, geo_t<8, 256>>, D>(C, batch, stream, "mfma_f8")
                    : chain_go<f8_mma_t<0, 0, geo_t<4, 128>>, D>(C, batch, stream, "mfma_f8");
    };
    if (C.split > 1) return chain_go_parts<f8_mma_t<0, 0, geo_t<4, 128>>>(dst_dt, C, batch, stream, "mfma_f8");
    if (dst_dt == MI355_DT_BF16) return go(std::integral_constant<int, CHAIN_BF16> {});
    if (dst_dt == MI355_DT_F32) return go(std::integral_constant<int, CHAIN_F32> {});
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
