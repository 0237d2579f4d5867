// Small products of 16-bit, fp8 and block-scaled operands on the chain epilogue: 32 x 32 tiles, as chain_small_kernel
// (kern_chain_i8.hip) has them for int8.
//
// A launch of a few 256 x 128 tiles is a chain of latencies -- 13 us for a product of 12 steps of K: ring, barriers,
// an epilogue of 64 values a lane.  Here a workgroup of four wavefronts owns 32 x 32 of dst, the wavefronts take the steps of 128
// bytes of K in turn, operands come straight from memory into the fragments (whole lines: chunks q and 4 + q of a row to
// lane (row, q), as in the large tiles), SD steps ahead, and the four partial tiles meet in LDS; a thread then owns four columns
// of a row, whose scales, bias and second tensor were asked for together with the first steps.  Block scales are read
// where they lie, a byte a lane, block and fragment: no pre-pass.
// Bound: latency while the tiles are no more than the CUs, then the operands' way through the L1s, which every tile
// repeats: 32 rows of either a step for 32 x 32 products.
#define MI355_CHAIN_KERNELS
#include "chain_gemm.hpp"
#include "line_policies.hpp"

namespace mi355 {
namespace {
constexpr int FST = 32, FSNW = 4;
constexpr long SMALL_MXF8_PARTS = 256; // MXFP8: up to so many tiles K goes to the four wavefronts in parts

// KIND's policy of line_policies.hpp (the geometry is not used)
template <int KIND>
using small_mma_t = std::conditional_t<KIND == CHAIN_SMALL_BF16, h16x16_mma_t<true, geo_t<4, 128>>,
        std::conditional_t<KIND == CHAIN_SMALL_F16, h16x16_mma_t<false, geo_t<4, 128>>,
                std::conditional_t<KIND == CHAIN_SMALL_F8, f8_mma_t<0, 0, geo_t<4, 128>>,
                        std::conditional_t<KIND == CHAIN_SMALL_MXF8, mxf8_mma_t<0, 0, geo_t<4, 128>>, mxf4_mma_t<geo_t<4, 128>>>>>>;

// IN_ORDER: a wavefront owns 16 x 16 of the tile and all of K, in the large tiles' order of sums.
template <int KIND, int DST, bool IN_ORDER>
__global__ void __launch_bounds__(FSNW * 64, IN_ORDER ? 3 : KIND >= CHAIN_SMALL_MXF8 ? 2 : 4) chain_small_float_kernel(const chain_more_t C) {
    using Mma = small_mma_t<KIND>;
    constexpr int NU = Mma::NU, NS = Mma::SCALE_SETS; // instructions a pair; scales a lane, fragment and step
    // steps of a wavefront in flight (four, at half the workgroups a CU, took as long or up to 1.8 times as long: 512 x 2048 x 512
    // fp8 19.0 us against 10.7)
    constexpr int SD = IN_ORDER ? 3 : 2;
    constexpr int NF = IN_ORDER ? 1 : 2, STRIDE = IN_ORDER ? 1 : FSNW; // fragments of 16 rows a wavefront; its next step
    __shared__ float part[IN_ORDER ? 1 : FSNW][16][64];
    const int t = threadIdx.x, lane = t & 63, j = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const long b = blockIdx.z, M = C.M, N = C.N;
    const int kbytes = (int)C.kbytes;
    const long m0 = (long)(blockIdx.x / C.tiles_n) * FST, n0 = (long)(blockIdx.x % C.tiles_n) * FST;
    // rows and columns beyond the edge read the last valid one (never stored)
    const char *arow[NF], *bcol[NF];
    const uint8_t *asc[NF], *bsc[NF];
    const int kblocks = (int)C.kbytes * (KIND == CHAIN_SMALL_MXF4 ? 2 : 1) / 32;
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        const long m = min(m0 + 16 * (IN_ORDER ? wave >> 1 : i) + j, M - 1), n = min(n0 + 16 * (IN_ORDER ? wave & 1 : i) + j, N - 1);
        arow[i] = C.a + b * C.a_bs + m * C.lda;
        bcol[i] = C.bt + b * C.b_bs + n * C.ldb;
        if constexpr (NS > 0) {
            asc[i] = C.sa + b * C.sa_bs + m * kblocks;
            bsc[i] = C.sb + b * C.sb_bs + n;
        }
    }
    struct step_t {
        line_pair_t a[NF], b[NF];
        int sa[NF][NS ? NS : 1], sb[NF][NS ? NS : 1];
    };
    // kbytes is a multiple of 16: a chunk is inside K or beyond it.  Those beyond are loaded from the row's last one and zeroed
    // in both operands before they are multiplied (a branch around the load would be a wait for everything in flight).
    auto load = [&](int s) __attribute__((always_inline)) {
        step_t f;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = min(s * 128 + 64 * u + 16 * q, kbytes - 16);
#pragma unroll
            for (int i = 0; i < NF; ++i) {
                f.a[i].c[u] = *(const v4i *)(arow[i] + k);
                f.b[i].c[u] = *(const v4i *)(bcol[i] + k);
            }
        }
        if constexpr (NS > 0) {
#pragma unroll
            for (int u = 0; u < NS; ++u) {
                const int blk = min(s * (4 * NS) + 4 * u + q, kblocks - 1);
#pragma unroll
                for (int i = 0; i < NF; ++i) {
                    f.sa[i][u] = asc[i][blk];
                    f.sb[i][u] = bsc[i][(unsigned)blk * (unsigned)N];
                }
            }
        }
        return f;
    };
    const int nsteps = (kbytes + 127) / 128;
    int step = IN_ORDER ? 0 : wave;
    step_t st[SD];
#pragma unroll
    for (int d = 0; d < SD; ++d) {
        const int sl = step + d * STRIDE;
        st[d] = load(sl < nsteps ? sl : 0);
    }
    // this thread's four outputs
    const int ui = wave >> 1, ujn = wave & 1;
    const long m = m0 + 16 * ui + j, n = n0 + 16 * ujn + 4 * q;
    chain_quad_t<DST> Q;
    if (m < M && n < N) Q.load(C, b, m, n);

    v4f acc[NF][NF];
#pragma unroll
    for (int i = 0; i < NF; ++i)
#pragma unroll
        for (int jn = 0; jn < NF; ++jn) acc[i][jn] = v4f {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](step_t &f, int s) __attribute__((always_inline)) {
        if (s * 128 + 128 > kbytes) { // (uniform: the last, partial step)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int keep = s * 128 + 64 * u + 16 * q < kbytes ? -1 : 0;
#pragma unroll
                for (int i = 0; i < NF; ++i) f.a[i].c[u] &= keep, f.b[i].c[u] &= keep;
            }
        }
        static_for<NU>([&](auto U) __attribute__((always_inline)) {
            constexpr int su = NS > 1 ? decltype(U)::value : 0;
#pragma unroll
            for (int i = 0; i < NF; ++i)
#pragma unroll
                for (int jn = 0; jn < NF; ++jn)
                    Mma::template mma<0, 0>(acc[i][jn], f.b[jn], f.a[i], U, NS ? f.sb[jn][su] : 0, NS ? f.sa[i][su] : 0);
        });
    };
    for (; step + (SD - 1) * STRIDE < nsteps; step += SD * STRIDE) {
#pragma unroll
        for (int d = 0; d < SD; ++d) {
            multiply(st[d], step + d * STRIDE);
            const int sl = step + (SD + d) * STRIDE;
            if (sl < nsteps) st[d] = load(sl); // (uniform over the wavefront)
        }
    }
#pragma unroll
    for (int d = 0; d < SD; ++d)
        if (step + d * STRIDE < nsteps) multiply(st[d], step + d * STRIDE);
    float x[4];
    if constexpr (IN_ORDER) {
        if (m >= M || n >= N) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = acc[0][0][e];
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int jn = 0; jn < 2; ++jn)
#pragma unroll
                for (int e = 0; e < 4; ++e) part[wave][i * 8 + jn * 4 + e][lane] = acc[i][jn][e];
        __syncthreads();
        if (m >= M || n >= N) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = part[0][ui * 8 + ujn * 4 + e][lane];
#pragma unroll
            for (int w = 1; w < FSNW; ++w) x[e] += part[w][ui * 8 + ujn * 4 + e][lane];
        }
    }
    Q.finish(C, b, m, n, x);
}
} // namespace

bool small_tiles_fit(long M, long N, long kbytes, int mx) {
    return kbytes < (1L << 30) && (M + FST - 1) / FST * ((N + FST - 1) / FST) < (1L << 31)
            && (mx == 0 || kbytes * 8 / mx / 32 * N < (1L << 32));
}

// Both sides in ns.  Small / 256 x 128 tiles, K split where that pays, us, launches after each other on the same operands: fp8 16 x
// 2240 x 1024 4.1 / 12.7, 256 x 2048 x 1024 6.3 / 13.5, 64 x 4096 x 4096 10.3 / 16.2, but 64 x 640 x 16384 30.1 / 15.9; bf16 32 x 1792 x 768
// 5.1 / 13.8, 512 x 1024 x 1024 9.7 / 16.2, 128 x 1024 x 8192 (f16) 30.4 / 16.1, 512 x 3600 x 704 23.1 / 14.7; MXFP4 128 x 2048 x 2048 5.4 / 18.4
// (whose 7 us of pre-pass kernels it does without), MXFP8 240 x 1040 x 1056 7.1 / 20.7.  On 25 shapes the side taken is the faster or within 1.03 of
// it, but for fp8 300 x 1040 x 4096 (17.1 / 14.8).
// MXFP8 beyond 256 tiles, in the large tiles' order (data that tests/test_mxf8_gemm.py calls exact takes 25 bits there, so that its
// bits follow the order of the sums): 300 x 1040 x 1056 7.7 / 20.6, 128 x 3520 x 1408 13.2 / 20.1, 700 x 1024 x 640 9.8 / 17.1.
// A workgroup's steps are a chain (1.67 ns a byte of K), its neighbours' traffic comes on top (per tile).
bool small_tiles_float(long batch, long M, long N, long kbytes, const chain_split_t &split, long step_ns, const chain_t &C, int mx) {
    const double tiles = (double)((M + FST - 1) / FST) * ((N + FST - 1) / FST) * batch;
    if (tiles > 1024) return false;
    const double large = (double)((M + 255) / 256) * ((N + 127) / 128) * batch;
    const double small = mx == 8 && tiles > SMALL_MXF8_PARTS ? 3300 + 8.2 * kbytes + tiles * 9
                                                              : 3300 + 1.67 * kbytes + tiles * (3 + 0.0025 * kbytes);
    const double rest = (mx ? 7000 : 0) + (C.act >= CHAIN_GELU ? 3000 : 0)
            + (split.split > 1 ? 8000 + split.part_steps * step_ns + split.split * large * 35 : 8500 + (kbytes + 127) / 128 * 500.);
    return small < 0.95 * rest;
}

int chain_launch_small(chain_small_t kind, int dst_dt, chain_more_t &C, unsigned batch, hipStream_t stream) {
    const long tm = (C.M + FST - 1) / FST, tn = (C.N + FST - 1) / FST;
    C.tiles_m = (int)tm;
    C.tiles_n = (int)tn;
    auto go = [&](auto k, auto dst) -> int {
        constexpr int K = decltype(k)::value, D = decltype(dst)::value;
        const dim3 grid((unsigned)(tm * tn), 1, batch);
        if constexpr (K == CHAIN_SMALL_MXF8) {
            if (tm * tn * batch > SMALL_MXF8_PARTS) {
                hipLaunchKernelGGL((chain_small_float_kernel<K, D, true>), grid, dim3(FSNW * 64), 0, stream, C);
                return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
            }
        }
        hipLaunchKernelGGL((chain_small_float_kernel<K, D, false>), grid, dim3(FSNW * 64), 0, stream, C);
        return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
    };
    auto by_dst = [&](auto k) -> int {
        if (dst_dt == MI355_DT_BF16) return go(k, std::integral_constant<int, CHAIN_BF16> {});
        if (dst_dt == MI355_DT_F32) return go(k, std::integral_constant<int, CHAIN_F32> {});
        if (dst_dt == MI355_DT_F16) return go(k, std::integral_constant<int, CHAIN_F16> {});
        return MI355_UNIMPLEMENTED;
    };
    switch (kind) {
        case CHAIN_SMALL_BF16: return by_dst(std::integral_constant<int, CHAIN_SMALL_BF16> {});
        case CHAIN_SMALL_F16: return by_dst(std::integral_constant<int, CHAIN_SMALL_F16> {});
        case CHAIN_SMALL_F8: return by_dst(std::integral_constant<int, CHAIN_SMALL_F8> {});
        case CHAIN_SMALL_MXF8: return by_dst(std::integral_constant<int, CHAIN_SMALL_MXF8> {});
        case CHAIN_SMALL_MXF4: return by_dst(std::integral_constant<int, CHAIN_SMALL_MXF4> {});
    }
    return MI355_UNIMPLEMENTED;
}

} // namespace mi355
