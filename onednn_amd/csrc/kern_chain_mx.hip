// The block-scaled types (MXFP8 e4m3 x e4m3 of hip:mfma_f8, hip:mfma_mxf4) on the chain kernels (chain_gemm.hpp).
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {

int chain_launch_mx(bool fp4, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
    using wide_t = geo_t<8, 256>;
    using narrow_t = geo_t<4, 128>;
    auto go = [&](auto dst) -> int {
        constexpr int D = decltype(dst)::value;
        if (fp4)
            return wide ? chain_go<mxf4_mma_t<wide_t>, D>(C, batch, stream, "mfma_mxf4")
                        : chain_go<mxf4_mma_t<narrow_t>, D>(C, batch, stream, "mfma_mxf4");
        return wide ? chain_go<mxf8_mma_t<0, 0, wide_t>, D>(C, batch, stream, "mfma_f8")
                    : chain_go<mxf8_mma_t<0, 0, narrow_t>, D>(C, batch, stream, "mfma_f8");
    };
    if (C.split > 1)
        return fp4 ? chain_go_parts<mxf4_mma_t<narrow_t>>(dst_dt, C, batch, stream, "mfma_mxf4")
                   : chain_go_parts<mxf8_mma_t<0, 0, narrow_t>>(dst_dt, C, batch, stream, "mfma_f8");
    if (dst_dt == MI355_DT_BF16) return go(std::integral_constant<int, CHAIN_BF16> {});
    if (dst_dt == MI355_DT_F32) return go(std::integral_constant<int, CHAIN_F32> {});
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
