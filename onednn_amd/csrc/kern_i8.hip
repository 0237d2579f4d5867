// "hip:mfma_i8" -- LDS-tiled int8 GEMM on the gfx950 matrix cores
// (v_mfma_i32_16x16x64_i8, line_loops.hpp) with the zero-point compensation folded into an
// s32 row/column-sum correction and the reference's epilogue fused in.
//
// Replaces, for integer src and weights, the reference's brgemm int8 path
// (src/cpu/x64/matmul/brgemm_matmul.cpp:658-1027: copy_B with s8s8/zp
// compensation + AMX/VNNI microkernel + jit_brgemm_post_ops) and computes the
// same values as ref_matmul_int8_t (src/cpu/matmul/ref_matmul_int8.cpp:174-306)
// when there is a single group along K:
//   acc[m,n] = sum_k (src[m,k] - zs) * (wei[k,n] - zw[n])          (s32)
//            = sum_k s'w' + a*colsum'[n] + c[n]*rowsum'[m] + K*a*c[n]
//     with s' = src - off_s, w' = wei - off_w the bytes re-biased to s8
//     (off = 128 for u8, 0 for s8), a = off_s - zs, c[n] = off_w - zw[n];
//   d = (float)acc * src_scale * wei_scale[n]  -> shared epilogue.
#include "chain_gemm.hpp"
#include "line_policies.hpp"

#include <cstdlib>
#include <cstring>

namespace mi355 {

namespace {

using namespace gemm;
constexpr int BK = BKB;       // int8: one byte per K element
using i8_geo_t = geo_t<8, 256>;

struct i8_extra_t {
    const int8_t *bt; // weights as [N][K] bytes, K contiguous
    long ldb;         // bytes between consecutive n
    long bt_bstride;  // bytes between batches (0 = broadcast)
    const int *colsum; // [Bw][N] sum_k w'  (null when a == 0)
    const int *rowsum; // [Bs][M] sum_k s'  (null when c == 0)
    int tiles_m, tiles_n;
};

// raw s32 accumulator -> f32 entering the shared epilogue
struct i8_conv_t {
    typedef int row_t;
    float ssc;
    bool with_src_sc, with_wei_sc, has_comp;
    const int *rowsum; // already offset to this batch, or null
    const int *colsum; // already offset to this batch, or null
    int a_c, off_w, Kc;
    long bw;
    // the per-column operands of the table: weights scale, a * colsum'[n] + K a c[n], c[n]
    template <class PT>
    __device__ __forceinline__ void per_n(const PT &P, long, long n, float &wsc, int &cc, int &c) const {
        c = off_w;
        if (P.wei_zp.dt != MI355_DT_UNDEF)
            c -= load_int(P.wei_zp.dt, P.wei_zp.p, quant_off(P.wei_zp, bw, 0, n, P.K, P.N));
        cc = (a_c != 0 ? a_c * colsum[n] : 0) + Kc * a_c * c;
        if (with_wei_sc)
            wsc = load_float(P.wei_scale.dt, P.wei_scale.p, quant_off(P.wei_scale, bw, 0, n, P.K, P.N));
    }
    __device__ __forceinline__ int row_data(long m) const { return rowsum ? rowsum[m] : 0; }

    __device__ __forceinline__ void quad(const v4i_t &raw, int rs, unsigned ntab, int col, float (&f)[4]) const {
        int v[4] = {raw[0], raw[1], raw[2], raw[3]};
        if (has_comp) {
            const v4i_t cc = nt4i(ntab, NT_CC, col), c = nt4i(ntab, NT_C, col);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += cc[e] + c[e] * rs;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = (float)v[e];
        if (with_src_sc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] *= ssc;
        }
        if (with_wei_sc) {
            const v4f_t w = nt4f(ntab, NT_WSC, col);
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] *= w[e];
        }
    }
};

extern __shared__ __attribute__((aligned(128))) char i8_smem[];

template <bool SRC_U8, bool WEI_U8, class G>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(G::NW / 4))) i8_gemm_kernel(const problem_t P_, const i8_extra_t X) {
    using Mma = i8_mma_t<SRC_U8, WEI_U8, G>;
    const auto &P = MI355_KERNARG_PROBLEM();
    char *smem = i8_smem;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = G::wm(wave), wn = G::wn(wave);
    const long b = blockIdx.z;
    const tile_pos_t tp = tile_position<G>((int)blockIdx.x, X.tiles_m, X.tiles_n);
    const long m0 = tp.m0, n0 = tp.n0;

    const long lda = P.ss[1];
    const char *A = (const char *)P.src + (P.ss[0] ? b * P.ss[0] : 0) + m0 * lda;
    const char *Bt = (const char *)X.bt + b * X.bt_bstride + n0 * X.ldb;

    // ---- the epilogue's per-column operands go into their LDS table now: the
    // loads hide behind the pipeline prologue
    const long bs = P.ss[0] ? b : 0, bw = P.ws[0] ? b : 0;
    const int off_s = SRC_U8 ? 128 : 0, off_w = WEI_U8 ? 128 : 0;
    i8_conv_t cv;
    cv.a_c = off_s;
    if (P.src_zp.dt != MI355_DT_UNDEF) cv.a_c -= load_int(P.src_zp.dt, P.src_zp.p, 0);
    cv.off_w = off_w;
    cv.Kc = (int)P.K;
    cv.bw = bw;
    cv.with_src_sc = P.src_scale.dt != MI355_DT_UNDEF;
    cv.with_wei_sc = P.wei_scale.dt != MI355_DT_UNDEF;
    cv.ssc = cv.with_src_sc ? load_float(P.src_scale.dt, P.src_scale.p, 0) : 1.f;
    cv.rowsum = X.rowsum ? X.rowsum + bs * P.M : nullptr;
    cv.colsum = X.colsum ? X.colsum + bw * P.N : nullptr;
    cv.has_comp = X.rowsum != nullptr || X.colsum != nullptr || cv.a_c != 0 || WEI_U8 || P.wei_zp.dt != MI355_DT_UNDEF;
    const unsigned ntab = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem + line_loader_t<Mma>::LDS_BYTES;
    auto fill = [&]() __attribute__((always_inline)) { fill_ntab<G::NT>(P, cv, ntab, b, n0); };

    v4i acc[Mma::ROWS][Mma::COLS];
#pragma unroll
    for (int i = 0; i < Mma::ROWS; ++i)
#pragma unroll
        for (int j = 0; j < Mma::COLS; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;

    main_loop_lines<Mma>(acc, smem, A, Bt, lda, X.ldb, P.M - m0, P.N - n0, P.K, line_scales_t {}, fill);

    store_quadrant<layout16_t, G::WCOLS>(P, smem, ntab, acc, b, m0 + wm * 128, n0 + wn * G::WCOLS, wn * G::WCOLS, cv);
}


// ---- few tiles: 32 x 32 dst tiles
// without LDS staging.  The 256 x 256 tiles above leave the device idle when
// M x N holds only a handful of them (4 workgroups for 256 x 1024).  Here a workgroup of four wavefronts owns a
// 32 x 32 tile, the wavefronts take every fourth 64-byte step of K, each lane
// loads its MFMA operands (16 bytes of a src row, 16 bytes of a weights
// column, K contiguous in both) straight from memory, four steps ahead of the
// matrix cores, and a step beyond K's last 16 bytes is filled with the
// operand's zero.  The column sums of the weights and the row sums of src that
// the zero-point correction needs come out of two more MFMAs per operand tile
// against all-ones bytes, in the accumulators' own lane layout: no pre-pass
// kernels.  The four wavefronts' sums are added through LDS in wavefront order
// (integer: exact in any order), converted like the large tiles' and finished
// by the general epilogue.
constexpr int ST = 32;     // rows and columns of a small tile
constexpr int SNW = 4;     // wavefronts of its workgroup

template <bool SRC_U8, bool WEI_U8>
__global__ void __launch_bounds__(SNW * 64) i8_small_kernel(const problem_t P_, const i8_extra_t X) {
    // [wavefront][slot][lane]; slots: 16 accumulators, 8 column sums, 8 row sums
    __shared__ int part[SNW][32][64];
    const auto &P = MI355_KERNARG_PROBLEM();
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int j = lane & 15, q = lane >> 4;
    const long b = blockIdx.z;
    const long m0 = (long)(blockIdx.x / X.tiles_n) * ST, n0 = (long)(blockIdx.x % X.tiles_n) * ST;
    const long M = P.M, N = P.N, K = P.K;
    const long lda = P.ss[1];
    const char *A = (const char *)P.src + (P.ss[0] ? b * P.ss[0] : 0);
    const char *Bt = (const char *)X.bt + b * X.bt_bstride;
    // rows and columns beyond the edge read the last valid one (never stored)
    const char *arow[2], *bcol[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const long m = m0 + 16 * i + j < M ? m0 + 16 * i + j : M - 1;
        const long n = n0 + 16 * i + j < N ? n0 + 16 * i + j : N - 1;
        arow[i] = A + m * lda + 16 * q;
        bcol[i] = Bt + n * X.ldb + 16 * q;
    }
    const int a_fill = SRC_U8 ? (int)0x80808080 : 0, b_fill = WEI_U8 ? (int)0x80808080 : 0;
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
            f.b[i] = v4i {b_fill, b_fill, b_fill, b_fill};
            if (in) {
                f.a[i] = *(const v4i *)(arow[i] + k);
                f.b[i] = *(const v4i *)(bcol[i] + k);
            }
        }
        return f;
    };
    v4i acc[2][2], cs[2], rs[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        cs[i] = rs[i] = v4i {0, 0, 0, 0};
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) acc[i][jn] = v4i {0, 0, 0, 0};
    }
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const long nsteps = (K + 63) / 64;
    // SD of the wavefront's steps are in flight: a launch of a few hundred tiles lasts a handful of memory
    // latencies, and with one step ahead every step of a wavefront cost one of them
    constexpr int SD = 4;
    auto multiply = [&](const frag_t &cur) __attribute__((always_inline)) {
        v4i a[2], w[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            a[i] = SRC_U8 ? (cur.a[i] ^ (int)0x80808080) : cur.a[i];
            w[i] = WEI_U8 ? (cur.b[i] ^ (int)0x80808080) : cur.b[i];
        }
        // operands exchanged as in the large tiles: a lane holds four
        // consecutive n (4 * (lane / 16) + e) of row lane % 16
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int jn = 0; jn < 2; ++jn)
                acc[i][jn] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[jn], a[i], acc[i][jn], 0, 0, 0);
            cs[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], ones, cs[i], 0, 0, 0); // [e]: column 4 * (lane / 16) + e
            rs[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, a[i], rs[i], 0, 0, 0); // every e: row lane % 16
        }
    };
    long step = wave;
    frag_t st[SD];
#pragma unroll
    for (int d = 0; d < SD; ++d) {
        const long sl = step + (long)d * SNW;
        st[d] = load(sl < nsteps ? sl : 0);
    }
    for (; step + (long)(SD - 1) * SNW < nsteps; step += (long)SD * SNW) {
#pragma unroll
        for (int d = 0; d < SD; ++d) {
            multiply(st[d]);
            const long sl = step + (long)(SD + d) * SNW;
            if (sl < nsteps) st[d] = load(sl); // (uniform over the wavefront)
        }
    }
#pragma unroll
    for (int d = 0; d < SD; ++d)
        if (step + (long)d * SNW < nsteps) multiply(st[d]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int jn = 0; jn < 2; ++jn) part[wave][i * 8 + jn * 4 + e][lane] = acc[i][jn][e];
            part[wave][16 + i * 4 + e][lane] = cs[i][e];
            part[wave][24 + i * 4 + e][lane] = rs[i][e];
        }
    }
    __syncthreads();
    // thread (unit = i, jn; lane): the quad of row m0 + 16 i + lane % 16,
    // columns n0 + 16 jn + 4 (lane / 16) ..
    const int unit = t >> 6, ui = unit >> 1, ujn = unit & 1;
    int sum[4] = {0, 0, 0, 0}, csum[4] = {0, 0, 0, 0}, rsum = 0;
#pragma unroll
    for (int wv = 0; wv < SNW; ++wv) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sum[e] += part[wv][ui * 8 + ujn * 4 + e][lane];
            csum[e] += part[wv][16 + ujn * 4 + e][lane];
        }
        rsum += part[wv][24 + ui * 4][lane];
    }
    const long m = m0 + 16 * ui + j, nbase = n0 + 16 * ujn + 4 * q;
    if (m >= M || nbase >= N) return;
    const int nvalid = N - nbase < 4 ? (int)(N - nbase) : 4;
    const long bw = P.ws[0] ? b : 0;
    int a_c = SRC_U8 ? 128 : 0;
    if (P.src_zp.dt != MI355_DT_UNDEF) a_c -= load_int(P.src_zp.dt, P.src_zp.p, 0);
    const bool with_src_sc = P.src_scale.dt != MI355_DT_UNDEF, with_wei_sc = P.wei_scale.dt != MI355_DT_UNDEF;
    const float ssc = with_src_sc ? load_float(P.src_scale.dt, P.src_scale.p, 0) : 1.f;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (e < nvalid) {
            const long n = nbase + e;
            int c = WEI_U8 ? 128 : 0;
            if (P.wei_zp.dt != MI355_DT_UNDEF)
                c -= load_int(P.wei_zp.dt, P.wei_zp.p, quant_off(P.wei_zp, bw, 0, n, P.K, P.N));
            // the large tiles' order: a * colsum + K * a * c, then + c * rowsum
            const int cc = a_c * csum[e] + (int)K * a_c * c;
            float f = (float)(sum[e] + (cc + c * rsum));
            if (with_src_sc) f *= ssc;
            if (with_wei_sc)
                f *= load_float(P.wei_scale.dt, P.wei_scale.p, quant_off(P.wei_scale, bw, 0, n, P.K, P.N));
            v[e] = f;
        }
    }
    apply_epilogue4(P, v, b, m, nbase, nvalid);
    store4(P, P.ds[2] == 1 && vec_ok_store(P.dst, P.ds[0], P.ds[1], dt_bits(P.dst_dt)), v, b, m, nbase, nvalid);
}

// out[b][r] = sum_k (bytes[b][r][k] ^ flip) as signed bytes; one wave per row
__global__ void __launch_bounds__(256) i8_rowsum_kernel(const int8_t *p, long rows, long K,
        long ld, long bs, int flip, int *out) {
    p += blockIdx.y * bs;
    out += blockIdx.y * rows;
    const long r = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    const int8_t *row = p + r * ld;
    int s = 0;
    const long k16 = K / 16 * 16;
    for (long k = lane * 16; k < k16; k += 64 * 16) {
        v4i v = *(const v4i *)(row + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int w = v[i] ^ flip;
            s += (int)(int8_t)(w & 0xff) + (int)(int8_t)((w >> 8) & 0xff)
                    + (int)(int8_t)((w >> 16) & 0xff) + (w >> 24);
        }
    }
    for (long k = k16 + lane; k < K; k += 64) s += (int)(int8_t)(row[k] ^ (flip & 0xff));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
    if (lane == 0) out[r] = s;
}

struct i8_plan_t {
    bool small; // 32 x 32 tiles
    bool need_transpose, need_colsum, need_rowsum;
    size_t off_bt, off_colsum, off_rowsum, off_parts, total;
    chain_split_t split; // of K on the LDS tiles, where the scratch has room for the parts
    long Bw, Bs;
};

// The epilogue as a chain of chain_gemm.hpp that the int8 kernels have, as far as the descriptor tells (where dst lies is the
// launch's to look at); false: the general kernels.
bool i8_chain(const problem_t &P, chain_t &C) {
    return P.wei_dt == MI355_DT_S8 && P.wei_zp.dt == MI355_DT_UNDEF && (P.src_zp.dt == MI355_DT_UNDEF || P.src_zp.dt == MI355_DT_S32)
            && P.dst_dt != MI355_DT_F16 && chain_form(P, true, false, C);
}

// The small tiles' time grows with their number, the LDS tiles' -- up to 128 of them -- hardly at all, so the line between
// the two is a number of small tiles.  (Not of large ones: a short M fills few rows of a large tile.)  What moves it, with
// small against LDS tiles in us:
//   K       1024 tiles (256 x 4096, s8 -> s8 with K = 1024 / 4096 / 16384): 10.7 / 14.5, 31.5 / 26.0, 115 / 74
//   a K of no whole 128-byte lines: the small tiles' rows then start in different channels, and the LDS tiles have a
//           partial last step (the same with K = 1040 / 4112 / 16400): 8.8 / 15.4, 25.4 / 27.2, 89 / 107.  (Sums: 64 bytes.)
//   sums    that are kernels of their own in front of the LDS tiles (u8 -> bf16, 256 x 4096 x 4096): 31.9 / 34.8 against 31.5 /
//           26.0 without
//   the general epilogue, 4 us of a launch of small tiles and 8 to 12 of LDS tiles (f16 dst, 256 x 6144 x 1024): 21.5 /
//           23.5 against 14.4 / 14.7 of a chain
//   few rows: an LDS tile is seven eighths empty or more (16 x 65536 x 1024, s8 -> s8): 18.2 / 23.1 against 18.1 / 14.7 for 256 x
//           8192; with sums, whose time follows N, up to 64 of them (64 x 40960 x 2064, u8 -> bf16): 36.8 / 53.8
// The lines lie where the two meet in a grid of 26 K x 8 M x 11 numbers of tiles x 4 epilogues, the lowest over the M of a
// row; the choice is within 1.1 times the better one's time nearly everywhere.
bool small_tiles_better(const mi355_matmul_desc_t &d, bool chain) {
    constexpr int ALL = 1 << 30;
    static const int line[2][2][2][2][5] = {
            // [few rows][whole lines of K][general epilogue][sums][K < 512, < 2048, < 4096, < 8192, longer]
            {{{{1665, 2049, 1537, 1025, 1025}, {2561, 3073, 2049, 1537, 1153}}, {{1665, 2049, 1537, 1281, 1025}, {2561, 2561, 2049, 1537, 1153}}},
                    {{{769, 1281, 897, 641, 513}, {1281, 1793, 1281, 1025, 769}}, {{1281, 1537, 1025, 769, 641}, {1537, 2049, 1537, 1153, 769}}}},
            {{{{ALL, ALL, ALL, 2049, 1153}, {ALL, ALL, ALL, 2561, 2049}}, {{ALL, ALL, ALL, 2049, 1153}, {ALL, ALL, ALL, 2561, 1281}}},
                    {{{897, ALL, ALL, 1025, 769}, {1024, ALL, 2561, 1537, 1025}}, {{1025, ALL, ALL, 1025, 769}, {3073, ALL, ALL, 1537, 1025}}}}};
    const bool sums = d.src_dt == MI355_DT_U8 || d.wei_dt == MI355_DT_U8 || !quant_absent(d.src_zp) || !quant_absent(d.wei_zp);
    const int band = d.K < 512 ? 0 : d.K < 2048 ? 1 : d.K < 4096 ? 2 : d.K < 8192 ? 3 : 4;
    const bool few = d.M <= (chain && sums ? 64 : 32), whole = d.K % (sums ? BK : LKB) == 0;
    return ((d.M + ST - 1) / ST) * ((d.N + ST - 1) / ST) * d.batch < line[few][whole][!chain][sums][band];
}

// The line of small_tiles_better is drawn against LDS tiles that take all of K; with K split (chain_gemm.hpp) they are the better
// ones from fewer small tiles on where K is long.  Both sides in ns: 128 x 4096 x 4096 17.1 us small, 20.2
// split, 1024 x 1024 x 4096 31 and 20.3, 300 x 2048 x 8192 45.4 and 20.2, with sums 64 x 2048 x 16384 31.0 and 33.4, 415 x 1664 x 13024
// 56.1 and 34.2; a tenth in favour of the small tiles, one launch.
bool split_tiles_better(const mi355_matmul_desc_t &d, const chain_split_t &s) {
    const bool sums = d.src_dt == MI355_DT_U8 || !quant_absent(d.src_zp);
    const double small_tiles = (double)((d.M + ST - 1) / ST) * ((d.N + ST - 1) / ST) * d.batch;
    const double tiles = (double)((d.M + 255) / 256) * ((d.N + 127) / 128) * d.batch;
    const double small = 3500 + (small_tiles < 256 ? 256 : small_tiles) * d.K * (d.K % LKB == 0 ? 6.6e-3 : 5.2e-3);
    const double split = 9000 + s.part_steps * 700. + s.split * tiles * 52 + (sums ? 3500 + (double)d.N * d.K * 1e-4 : 0);
    return 1.1 * split < small;
}
// (the LDS tiles' offsets from a tile's first row are 32-bit, the small tiles' are not)
bool rows_fit_lds_tiles(const mi355_matmul_desc_t &d) {
    return d.src_stride[1] <= (1L << 24) && (d.wei_stride[1] == 1 ? d.wei_stride[2] : d.K) <= (1L << 24);
}
constexpr long I8_STEP_NS = 700; // of a 256 x 128 tile (chain_split)

// chain: what i8_chain says, the same of the descriptor's problem and of the launch's
i8_plan_t make_plan(const mi355_matmul_desc_t &d, bool chain, bool parts) {
    i8_plan_t p {};
    p.Bw = d.wei_stride[0] ? d.batch : 1;
    p.Bs = d.src_stride[0] ? d.batch : 1;
    p.need_transpose = !(d.wei_stride[1] == 1);
    p.small = !d.dst_scale_dynamic && small_tiles_better(d, chain);
    // the MI355_I8_TILES switch overrides the choice where both can run (tests and
    // tuning): large = the LDS tiles, 256 x 128 or 256 x 256 by the number of
    // tiles; wide = the 256 x 256 ones
    const int force = tuning(TUNE_I8_TILES);
    if (force == TUNE_LARGE || force == TUNE_WIDE || force == TUNE_NARROW) p.small = false;
    if (force == TUNE_SMALL && !d.dst_scale_dynamic) p.small = true;
    p.split = chain_split_t {1, 0};
    if (chain && parts && force == TUNE_AUTO) {
        const chain_split_t split = chain_split(d.batch, d.M, d.N, d.K, false, I8_STEP_NS);
        if (p.small && split.split > 1 && rows_fit_lds_tiles(d) && split_tiles_better(d, split)) p.small = false;
        if (!p.small) p.split = split;
    }
    // a = off_s - zs can be non-zero whenever src is u8 or has a zero point;
    // c likewise for the weights.  The small tiles compute their own sums: a
    // problem they run on K-contiguous weights needs no scratch at all.
    p.need_colsum = !p.small && (d.src_dt == MI355_DT_U8 || !quant_absent(d.src_zp));
    p.need_rowsum = !p.small && (d.wei_dt == MI355_DT_U8 || !quant_absent(d.wei_zp));
    // where a scratch buffer exists anyway its layout is that of the LDS tiles
    // (the sums are 4 (M + N) bytes), whichever tiles run
    const bool colsum = p.need_colsum || (p.need_transpose && (d.src_dt == MI355_DT_U8 || !quant_absent(d.src_zp)));
    const bool rowsum = p.need_rowsum || (p.need_transpose && (d.wei_dt == MI355_DT_U8 || !quant_absent(d.wei_zp)));
    size_t off = 0;
    p.off_bt = off;
    if (p.need_transpose) off += align_up((size_t)p.Bw * d.N * d.K, 256);
    p.off_colsum = off;
    if (colsum) off += align_up((size_t)p.Bw * d.N * 4, 256);
    p.off_rowsum = off;
    if (rowsum) off += align_up((size_t)p.Bs * d.M * 4, 256);
    p.off_parts = off;
    off += chain_parts_bytes(d.batch, d.M, d.N, false, p.split.split);
    p.total = off;
    return p;
}

} // namespace

int i8_supported(const mi355_matmul_desc_t &d) {
    if (!is_int8_dt(d.src_dt) || !is_int8_dt(d.wei_dt)) return MI355_UNIMPLEMENTED;
    if (dt_bits(d.dst_dt) < 8) return MI355_UNIMPLEMENTED;
    // whole 16-byte chunks of K
    if (d.K < 16 || d.K % 16 != 0) return MI355_UNIMPLEMENTED;
    if (d.K % BK != 0 && d.dst_scale_dynamic) return MI355_UNIMPLEMENTED;
    if (d.src_stride[2] != 1 || d.src_stride[1] % 16 != 0) return MI355_UNIMPLEMENTED;
    if (d.src_stride[0] % 16 != 0) return MI355_UNIMPLEMENTED;
    const bool k_major = d.wei_stride[1] == 1 && d.wei_stride[2] % 16 == 0
            && d.wei_stride[0] % 16 == 0;
    const bool n_major = d.wei_stride[2] == 1;
    if (!k_major && !n_major) return MI355_UNIMPLEMENTED;
    // single group along K, per-tensor src parameters, per-tensor or per-N
    // weights parameters
    if (!quant_absent(d.src_pr)) return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.src_scale) && (d.src_scale.mask != 0)) return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.src_zp) && (d.src_zp.mask != 0)) return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.wei_scale)
            && ((d.wei_scale.mask & 2) || d.wei_scale.group[0] > 1 || d.wei_scale.group[1] > 1))
        return MI355_UNIMPLEMENTED;
    if (!quant_absent(d.wei_zp)
            && ((d.wei_zp.mask & 2) || d.wei_zp.group[0] > 1 || d.wei_zp.group[1] > 1))
        return MI355_UNIMPLEMENTED;
    if (d.batch > 65535) return MI355_UNIMPLEMENTED;
    return MI355_SUCCESS;
}

bool i8_scratch_optional(const mi355_matmul_desc_t &d) { return d.K % BK != 0 && d.wei_stride[1] == 1; }

size_t i8_scratch_bytes(const mi355_matmul_desc_t &d, bool parts, size_t *fixed) {
    problem_t P;
    problem_of_desc(d, P);
    chain_t C;
    const i8_plan_t p = make_plan(d, i8_chain(P, C), parts);
    *fixed = p.off_parts;
    return p.total;
}

int i8_launch(const mi355_matmul_desc_t &d, const problem_t &P, const scratch_t &S, hipStream_t stream) {
    void *const scratch = S.p;
    chain_more_t C {};
    bool chain = i8_chain(P, C);
    i8_plan_t plan = make_plan(d, chain, S.split);
    const uintptr_t at = (uintptr_t)P.src | (plan.need_transpose ? 0 : (uintptr_t)P.wei);
    // K is split on the LDS tiles, whose loads bring whole chunks from 16-byte boundaries straight to LDS: operands off one
    // have the tiles that they have without parts, the small ones where those are the better ones
    if (plan.split.split > 1 && (at & 15)) plan = make_plan(d, chain, false);
    // A K that ends inside 64 bytes also takes operands off 16-byte boundaries, which the LDS tiles' loads cannot, and
    // K-contiguous weights without scratch: the small tiles'.
    if (!plan.small && d.K % BK != 0) {
        const bool without = plan.total > 0 && !scratch && i8_scratch_optional(d);
        if ((at & 15) || without) plan.small = true, plan.need_colsum = plan.need_rowsum = false;
        if (without) plan.total = 0;
    }
    if (plan.total > 0 && !scratch) {
        set_error("mfma_i8: %zu bytes of scratch required", plan.total);
        return MI355_INVALID_ARGUMENTS;
    }
    char *sc = (char *)scratch;
    i8_extra_t X {};
    const bool src_u8 = d.src_dt == MI355_DT_U8, wei_u8 = d.wei_dt == MI355_DT_U8;
    if (plan.need_transpose) {
        uint8_t *bt = (uint8_t *)(sc + plan.off_bt);
        transpose_bytes(P.wei, d.K, d.N, d.wei_stride[1], d.wei_stride[0], bt, d.K, d.N * d.K,
                plan.Bw, stream);
        X.bt = (const int8_t *)bt;
        X.ldb = d.K;
        X.bt_bstride = plan.Bw > 1 ? d.N * d.K : 0;
    } else {
        X.bt = (const int8_t *)P.wei;
        X.ldb = d.wei_stride[2];
        X.bt_bstride = d.wei_stride[0];
    }
    if (plan.need_colsum) {
        int *cs = (int *)(sc + plan.off_colsum);
        hipLaunchKernelGGL(i8_rowsum_kernel, dim3((unsigned)((d.N + 3) / 4), (unsigned)plan.Bw), dim3(256), 0, stream, X.bt, d.N,
                d.K, X.ldb, X.bt_bstride, wei_u8 ? (int)0x80808080 : 0, cs);
        X.colsum = cs;
    }
    if (plan.need_rowsum) {
        int *rs = (int *)(sc + plan.off_rowsum);
        hipLaunchKernelGGL(i8_rowsum_kernel, dim3((unsigned)((d.M + 3) / 4), (unsigned)plan.Bs), dim3(256), 0, stream,
                (const int8_t *)P.src, d.M, d.K, d.src_stride[1], d.src_stride[0], src_u8 ? (int)0x80808080 : 0, rs);
        X.rowsum = rs;
    }
    const bool su = d.src_dt == MI355_DT_U8, wu = d.wei_dt == MI355_DT_U8;
    chain = chain && chain_dst_aligned(C, P.dst_dt);
    if (chain) {
        C.a = (const char *)P.src; C.lda = P.ss[1]; C.a_bs = P.ss[0];
        C.bt = (const char *)X.bt; C.ldb = X.ldb; C.b_bs = X.bt_bstride;
        C.kbytes = P.K;
        C.colsum = X.colsum;
        C.colsum_bs = plan.Bw > 1 ? d.N : 0;
        C.src_zp = P.src_zp.dt != MI355_DT_UNDEF ? (const int *)P.src_zp.p : nullptr;
        C.off_s = su ? 128 : 0;
        C.parts = S.parts ? (char *)S.parts : sc + plan.off_parts;
        C.split = plan.split.split;
        C.part_steps = plan.split.part_steps;
    }
    if (plan.small) {
        if (chain) {
            const int st = chain_launch_i8_small(su, P.dst_dt, C, (unsigned)d.batch, stream);
            if (st != MI355_UNIMPLEMENTED) return st;
        }
        if (general_refused("mfma_i8")) return MI355_UNIMPLEMENTED;
        X.tiles_m = (int)((d.M + ST - 1) / ST);
        X.tiles_n = (int)((d.N + ST - 1) / ST);
        const long tiles = (long)X.tiles_m * X.tiles_n;
        if (tiles >= (1L << 31)) {
            set_error("mfma_i8: %ld small tiles exceed the grid", tiles);
            return MI355_UNIMPLEMENTED;
        }
        const dim3 sgrid((unsigned)tiles, 1, (unsigned)d.batch);
        auto go_small = [&](auto kern) -> int {
            hipLaunchKernelGGL(kern, sgrid, dim3(SNW * 64), 0, stream, P, X);
            return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
        };
        if (su && wu) return go_small(i8_small_kernel<true, true>);
        if (su) return go_small(i8_small_kernel<true, false>);
        if (wu) return go_small(i8_small_kernel<false, true>);
        return go_small(i8_small_kernel<false, false>);
    }
    // (MI355_I8_TILES: wide / narrow keep one geometry whatever the size: tests, tuning)
    const int force = tuning(TUNE_I8_TILES);
    const bool narrow = force == TUNE_NARROW || (line_tiles_narrow(d.batch, d.M, d.N, d.K, chain) && force != TUNE_WIDE);
    if (chain) {
        const int st = chain_launch_i8(su, P.dst_dt, C, (unsigned)d.batch, !narrow, stream);
        if (st != MI355_UNIMPLEMENTED) return st;
    }
    if (general_refused("mfma_i8")) return MI355_UNIMPLEMENTED;
    X.tiles_m = (int)((d.M + BM - 1) / BM);
    auto go = [&](auto su_, auto wu_) -> int {
        constexpr bool SU = decltype(su_)::value, WU = decltype(wu_)::value;
        auto run = [&](auto geo) -> int {
            using G = decltype(geo);
            constexpr int smem_bytes = line_loader_t<i8_mma_t<SU, WU, G>>::LDS_BYTES + NTAB_BYTES;
            X.tiles_n = (int)((d.N + G::BN - 1) / G::BN);
            const dim3 grid((unsigned)(X.tiles_m * X.tiles_n), 1, (unsigned)d.batch);
            const auto kern = i8_gemm_kernel<SU, WU, G>;
            if (const int st = ensure_dynamic_lds((const void *)kern, smem_bytes, "mfma_i8")) return st;
            hipLaunchKernelGGL(kern, grid, dim3(G::NT), smem_bytes, stream, P, X);
            return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
        };
        return narrow ? run(geo_t<4, 128> {}) : run(i8_geo_t {});
    };
    if (su && wu) return go(std::true_type {}, std::true_type {});
    if (su) return go(std::true_type {}, std::false_type {});
    if (wu) return go(std::false_type {}, std::true_type {});
    return go(std::false_type {}, std::false_type {});
}

} // namespace mi355
