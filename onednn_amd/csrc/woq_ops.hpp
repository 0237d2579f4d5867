// What the two decode kernels with 4-bit weights do in the activations' type: OFFSET + nibble, exact in either type,
// and the product.
#pragma once
#include "kernels.hpp"

namespace mi355 {

template <bool F16>
struct woq_ops_t {
    typedef int v4i __attribute__((ext_vector_type(4)));
    typedef float v4f __attribute__((ext_vector_type(4)));
    typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
    typedef _Float16 v8h __attribute__((ext_vector_type(8)));
    static constexpr float OFFSET = F16 ? 64.f : 128.f;
    static constexpr unsigned MAGIC = F16 ? 0x54005400u : 0x43004300u; // OFFSET, twice
    static constexpr int ONES = F16 ? 0x3C003C00 : 0x3F803F80;
    // the nibbles u and u + 4 of a dword: the last mantissa bits of a bf16 from 128 on are units, the fifth from the
    // end of an f16 from 64 on
    __device__ __forceinline__ static unsigned unpack(unsigned d, int u, unsigned magic) {
        if constexpr (F16) return ((u == 0 ? d << 4 : d >> (4 * u - 4)) & 0x00F000F0u) | magic;
        else return ((d >> (4 * u)) & 0x000F000Fu) | magic;
    }
    __device__ __forceinline__ static v4f mma(const v4i &a, const v4i &b, const v4f &c) {
        if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    }
};

// One element of dst from its terms, src (wei - zp) scale, one after the other.  Where src holds infinities the
// difference of two sums that the kernels take is NaN although the terms' sum may be an infinity: f16 activations, which
// overflow in earnest, come here then.  group: k per quantization group; nibble(k): the weight's bits, anything above them.
template <class XT, class F>
__device__ __forceinline__ float woq_term_sum(const XT &X, int group, int m, int n, F &&nibble) {
    const _Float16 *row = (const _Float16 *)X.src + (long)m * X.src_ld;
    float sum = 0.f;
#pragma unroll 1
    for (int k = 0; k < X.K && sum == sum; ++k) {
        const long g = (long)(k / group) * X.N;
        int w = (int)nibble(k) & 15;
        if (X.signed_w) w = (w ^ 8) - 8;
        const float zp = X.zp_dt == MI355_DT_UNDEF ? 0.f : (float)load_int(X.zp_dt, X.zp, X.zp_common ? 0 : (X.zp_grouped ? g : 0) + n);
        const float sc = X.sc_dt == MI355_DT_UNDEF ? 1.f : load_float(X.sc_dt, X.sc, (X.sc_grouped ? g : 0) + n);
        sum += (float)row[k] * (((float)w - zp) * sc);
    }
    return sum;
}

} // namespace mi355
