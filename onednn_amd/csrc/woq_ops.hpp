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

// Where f16 src holds infinities, which it does in earnest, the difference of two sums that the kernels take is NaN although
// the terms' sum may be an infinity.  A wavefront whose sums over its part of K, [k0, k1) in multiples of 16, are not finite
// takes them from those terms src (wei - zp) scale whose src or scale is not finite, next to which the others do not count: row m
// of src, a column n a lane, only lanes with `need` matter.  group: k per quantization group (a multiple of 16).
// Bound: a pass over the row's part, a latency per 512 elements, and one per eight that hold such a src.  N 8192, K 16384, packed /
// row-major, us: M 1 with an infinity 21 / 29 (finite 20 / 23; as a walk of every element along all of K 8200 / 11600), M 32 with
// one in every row 123 / 236 (finite 42 / 57; as walks 37700 / 40200).

// whether a scale of these columns is not finite
template <class XT>
__device__ __forceinline__ bool woq_bad_scales(const XT &X, int group, int n, int k0, int k1, bool need) {
    bool bad = false;
    if (X.sc_dt == MI355_DT_UNDEF) return false;
#pragma unroll 4
    for (int g = k0 / group; g <= (k1 - 1) / group; ++g)
        bad |= !__builtin_isfinite(load_float(X.sc_dt, X.sc, (X.sc_grouped ? (long)g * X.N : 0) + n));
    return __builtin_amdgcn_ballot_w64(need && bad) != 0;
}

// the sum; all: what woq_bad_scales said (every term is then looked up); nibble(k8, i): the bits of weight k8 + i (k8 a multiple of
// 8), anything above them
template <class XT, class F>
__device__ __forceinline__ float woq_term_sum(const XT &X, int group, int m, int n, int k0, int k1, bool all, bool need, F &&nibble) {
    const uint16_t *row = (const uint16_t *)X.src + (long)m * X.src_ld;
    const int lane = threadIdx.x & 63;
    float sum = 0.f;
    auto counts = [&](int k, unsigned x) __attribute__((always_inline)) {
        return __builtin_amdgcn_ballot_w64(k + lane < k1 && (all || (x & 0x7c00u) == 0x7c00u));
    };
#pragma unroll 1
    for (int k = k0; k < k1; k += 512) {
        unsigned xs[8], some = 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) xs[u] = row[min(k + 64 * u + lane, k1 - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u) some |= (counts(k + 64 * u, xs[u]) != 0 ? 1u : 0u) << u;
#pragma unroll 1
        for (; some != 0; some &= some - 1) {
            const int ku = k + 64 * __builtin_ctz(some);
            const unsigned x = row[min(ku + lane, k1 - 1)];
            unsigned long mask = counts(ku, x);
#pragma unroll 1
            for (int k8 = ku; mask != 0; k8 += 8, mask >>= 8) {
                if ((mask & 255) == 0) continue;
                const long gn = (long)(k8 / group) * X.N;
                const float zp = X.zp_dt == MI355_DT_UNDEF ? 0.f : (float)load_int(X.zp_dt, X.zp, X.zp_common ? 0 : (X.zp_grouped ? gn : 0) + n);
                const float sc = X.sc_dt == MI355_DT_UNDEF ? 1.f : load_float(X.sc_dt, X.sc, (X.sc_grouped ? gn : 0) + n);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    int w = (int)nibble(k8, i) & 15;
                    if (X.signed_w) w = (w ^ 8) - 8;
                    const uint16_t xi = (uint16_t)__builtin_amdgcn_readlane((int)x, k8 - ku + i);
                    const float term = (float)__builtin_bit_cast(_Float16, xi) * (((float)w - zp) * sc);
                    if ((mask >> i) & 1) sum += term;
                }
            }
            if (__builtin_amdgcn_ballot_w64(need && sum == sum) == 0) return sum; // (NaN whatever follows)
        }
    }
    return sum;
}

} // namespace mi355
