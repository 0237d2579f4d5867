// hip:mfma_f8's general kernel on 256 x 128 tiles of four wavefronts (line_tiles_narrow).  Kept apart from kern_f8.hip
// so that the two sets of instantiations compile side by side.
#include "f8_family.hpp"
#include "line_policies.hpp"

namespace mi355 {

int f8_launch_narrow(int fa, int fb, const problem_t &P, const char *bt, long ldb, long bt_bstride, unsigned batch, hipStream_t stream) {
    f8_extra_t X {};
    X.bt = bt;
    X.ldb = ldb;
    X.bt_bstride = bt_bstride;
    X.tiles_m = (int)((P.M + BM - 1) / BM);
    X.tiles_n = (int)((P.N + narrow_geo_t::BN - 1) / narrow_geo_t::BN);
    const dim3 grid((unsigned)(X.tiles_m * X.tiles_n), 1, batch);
    auto go = [&](auto mma) -> int {
        using Mma = decltype(mma);
        constexpr int smem_bytes = ring_of<Mma>::BYTES + NTAB_BYTES;
        const auto kern = f8_gemm_kernel<Mma>;
        if (const int st = ensure_dynamic_lds((const void *)kern, smem_bytes, "mfma_f8")) return st;
        hipLaunchKernelGGL(kern, grid, dim3(narrow_geo_t::NT), smem_bytes, stream, P, X);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    // fa / fb: 1 = e5m2, 0 = e4m3
    if (fa && fb) return go(f8_mma_t<1, 1, narrow_geo_t> {});
    if (fa) return go(f8_mma_t<1, 0, narrow_geo_t> {});
    if (fb) return go(f8_mma_t<0, 1, narrow_geo_t> {});
    return go(f8_mma_t<0, 0, narrow_geo_t> {});
}

} // namespace mi355
