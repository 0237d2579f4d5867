// hip:mfma_i8 on the chain kernels (chain_gemm.hpp).
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {
namespace {

// The 32 x 32 tiles of i8_small_kernel (kern_i8.hip: a workgroup of four wavefronts that take the 64-byte steps of K in
// turn, operands straight from memory, sums added through LDS) with a chain in place of the general epilogue.  Such a
// launch is a chain of latencies: one of memory for the operands, then, in the general kernel, one each for the zero
// point, the scales and the bias, and the instruction fetches of the interpreter behind them.  Here those operands are
// asked for together with the first steps'.  256 x 1024 x 1024, u8 -> f32: 8.9 -> 4.9 us.
constexpr int CST = 32, CSNW = 4;

template <bool SRC_U8, bool SUMS, int DST>
__global__ void __launch_bounds__(CSNW * 64) chain_small_kernel(const chain_t C) {
    constexpr int SLOTS = SUMS ? 24 : 16; // 16 accumulators, 8 column sums
    __shared__ int part[CSNW][SLOTS][64];
    const int t = threadIdx.x, lane = t & 63, j = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const long b = blockIdx.z, M = C.M, N = C.N, K = C.kbytes;
    const long m0 = (long)(blockIdx.x / C.tiles_n) * CST, n0 = (long)(blockIdx.x % C.tiles_n) * CST;
    const char *A = C.a + b * C.a_bs, *Bt = C.bt + b * C.b_bs;
    // rows and columns beyond the edge read the last valid one (never stored)
    const char *arow[2], *bcol[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        arow[i] = A + min(m0 + 16 * i + j, M - 1) * C.lda + 16 * q;
        bcol[i] = Bt + min(n0 + 16 * i + j, N - 1) * C.ldb + 16 * q;
    }
    const int a_fill = SRC_U8 ? (int)0x80808080 : 0;
    struct frag_t {
        v4i a[2], b[2];
    };
    // K is a multiple of 16: a lane's 16 bytes are inside K or beyond it
    auto load = [&](long step) __attribute__((always_inline)) {
        frag_t f;
        const long k = step * 64;
        const bool in = k + 16 * q < K;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            f.a[i] = v4i {a_fill, a_fill, a_fill, a_fill};
            f.b[i] = v4i {0, 0, 0, 0};
            if (in) {
                f.a[i] = *(const v4i *)(arow[i] + k);
                f.b[i] = *(const v4i *)(bcol[i] + k);
            }
        }
        return f;
    };
    constexpr int SD = 4; // steps of a wavefront in flight
    const long nsteps = (K + 63) / 64;
    long step = wave;
    frag_t st[SD];
#pragma unroll
    for (int d = 0; d < SD; ++d) {
        const long sl = step + (long)d * CSNW;
        st[d] = load(sl < nsteps ? sl : 0);
    }
    // what this thread's four outputs need: row m0 + 16 ui + j, columns nbase .. + 3
    const int ui = wave >> 1, ujn = wave & 1;
    const long m = m0 + 16 * ui + j, nbase = n0 + 16 * ujn + 4 * q;
    float w[4], bias[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const long n = min(nbase + e, N - 1);
        w[e] = C.wsc.dt != MI355_DT_UNDEF ? chain_load(C.wsc, b * C.wsc.bs + (C.wsc.per ? n : 0)) : 1.f;
        bias[e] = C.bias.dt != MI355_DT_UNDEF ? chain_load(C.bias, b * C.bias.bs + n) : 0.f;
    }
    const float ssc = C.ssc.dt != MI355_DT_UNDEF ? chain_load(C.ssc, b * C.ssc.bs) : 1.f;
    const int a_c = C.off_s - (C.src_zp ? *C.src_zp : 0);
    const float ds = C.ds_mode ? chain_load(chain_vec_t {C.dsc, C.dsc_dt, 0, 0}, 0) : 1.f;

    v4i acc[2][2], cs[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        cs[i] = v4i {0, 0, 0, 0};
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) acc[i][jn] = v4i {0, 0, 0, 0};
    }
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    auto multiply = [&](const frag_t &f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const v4i a = SRC_U8 ? (f.a[i] ^ (int)0x80808080) : f.a[i];
#pragma unroll
            for (int jn = 0; jn < 2; ++jn) acc[i][jn] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.b[jn], a, acc[i][jn], 0, 0, 0);
            if (SUMS) cs[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.b[i], ones, cs[i], 0, 0, 0); // [e]: column 4 q + e
        }
    };
    for (; step + (long)(SD - 1) * CSNW < nsteps; step += (long)SD * CSNW) {
#pragma unroll
        for (int d = 0; d < SD; ++d) {
            multiply(st[d]);
            const long sl = step + (long)(SD + d) * CSNW;
            if (sl < nsteps) st[d] = load(sl); // (uniform over the wavefront)
        }
    }
#pragma unroll
    for (int d = 0; d < SD; ++d)
        if (step + (long)d * CSNW < nsteps) multiply(st[d]);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int jn = 0; jn < 2; ++jn) part[wave][i * 8 + jn * 4 + e][lane] = acc[i][jn][e];
            if (SUMS) part[wave][16 + i * 4 + e][lane] = cs[i][e];
        }
    __syncthreads();
    if (m >= M || nbase >= N) return;
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        int sum = 0, csum = 0;
#pragma unroll
        for (int wv = 0; wv < CSNW; ++wv) {
            sum += part[wv][ui * 8 + ujn * 4 + e][lane];
            if (SUMS) csum += part[wv][16 + ujn * 4 + e][lane];
        }
        float f = (float)(sum + (SUMS ? a_c * csum : 0));
        f *= ssc;
        f *= w[e];
        if (C.bias.dt != MI355_DT_UNDEF) f += bias[e];
        if (C.act == CHAIN_RELU) {
            if (DST == CHAIN_I8) f = fmaxf(f, 0.f); // an integer dst turns NaN and -0 into 0 either way
            else f = f > 0 ? f : f * 0.f;
        }
        if (DST == CHAIN_I8 && C.ds_mode) f = C.ds_mode == 2 ? f * (1.f / ds) : f / ds;
        x[e] = f;
    }
    constexpr int SHIFT = DST == CHAIN_I8 ? 0 : DST == CHAIN_F32 ? 2 : 1;
    char *to = C.dst + b * C.dst_bs + m * C.dst_pitch + (nbase << SHIFT);
    const int nvalid = N - nbase < 4 ? (int)(N - nbase) : 4;
    if constexpr (DST == CHAIN_I8) {
        const unsigned word = pack4_i8(x, C.lo, C.hi);
        if (nvalid == 4) *(unsigned *)to = word;
        else
            for (int e = 0; e < nvalid; ++e) to[e] = (char)(word >> (8 * e));
    } else if constexpr (DST == CHAIN_F32) {
        if (nvalid == 4) *(v4f *)to = v4f {x[0], x[1], x[2], x[3]};
        else
#pragma unroll
            for (int e = 0; e < 3; ++e)
                if (e < nvalid) ((float *)to)[e] = x[e];
    } else {
        const unsigned h01 = f32_to_bf16(x[0]) | ((unsigned)f32_to_bf16(x[1]) << 16);
        const unsigned h23 = f32_to_bf16(x[2]) | ((unsigned)f32_to_bf16(x[3]) << 16);
        if (nvalid == 4) *(v2u_cell_t *)to = v2u_cell_t {h01, h23};
        else {
            ((uint16_t *)to)[0] = (uint16_t)h01;
            if (nvalid > 1) ((uint16_t *)to)[1] = (uint16_t)(h01 >> 16);
            if (nvalid > 2) ((uint16_t *)to)[2] = (uint16_t)h23;
        }
    }
}
} // namespace

int chain_launch_i8_small(bool src_u8, int dst_dt, chain_t &C, unsigned batch, hipStream_t stream) {
    const long tm = (C.M + CST - 1) / CST, tn = (C.N + CST - 1) / CST;
    if (tm * tn >= (1L << 31)) return MI355_UNIMPLEMENTED;
    C.tiles_m = (int)tm;
    C.tiles_n = (int)tn;
    auto go = [&](auto u8, auto sums, auto dst) -> int {
        hipLaunchKernelGGL((chain_small_kernel<decltype(u8)::value, decltype(sums)::value, decltype(dst)::value>),
                dim3((unsigned)(tm * tn), 1, batch), dim3(CSNW * 64), 0, stream, C);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    auto by_dst = [&](auto u8, auto sums) -> int {
        if (is_int8_dt(dst_dt)) return go(u8, sums, std::integral_constant<int, CHAIN_I8> {});
        if (dst_dt == MI355_DT_BF16) return go(u8, sums, std::integral_constant<int, CHAIN_BF16> {});
        if (dst_dt == MI355_DT_F32) return go(u8, sums, std::integral_constant<int, CHAIN_F32> {});
        return MI355_UNIMPLEMENTED;
    };
    if (src_u8) return by_dst(std::true_type {}, std::true_type {});
    return C.src_zp ? by_dst(std::false_type {}, std::true_type {}) : by_dst(std::false_type {}, std::false_type {});
}

int chain_launch_i8(bool src_u8, int dst_dt, chain_more_t &C, unsigned batch, bool wide, hipStream_t stream) {
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
    if (C.split > 1)
        return src_u8 ? chain_go_parts<i8_mma_t<true, false, geo_t<4, 128>>>(dst_dt, C, batch, stream, "mfma_i8")
                      : chain_go_parts<i8_mma_t<false, false, geo_t<4, 128>>>(dst_dt, C, batch, stream, "mfma_i8");
    return src_u8 ? by_dst(std::true_type {}) : by_dst(std::false_type {});
}

} // namespace mi355
