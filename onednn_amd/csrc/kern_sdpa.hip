// Scaled dot-product attention in one pass over the keys: dst = softmax(Q K * scale + mask) V for bf16 / f16 tensors of
// head size 64 or 128, without the scores ever leaving the registers (the composition of two matmuls around
// sdpa_softmax_kernel, kern_softmax.hip, writes and reads 12 bytes per score and stays for everything else).
//
// A wavefront owns 32 rows of queries and walks tiles of keys:
//   S^T = K Q^T   v_mfma_f32_32x32x16, keys as the first operand: a lane then holds one query's scores (column
//                 lane % 32, keys 8 (r / 4) + 4 (lane / 32) + r % 4), so the row maximum and sum are a reduction inside
//                 the lane and one exchange between the lane halves (v_permlane32_swap)
//   P^T           exp2 of the scores relative to the running maximum, packed in place: eight consecutive registers are
//                 the second operand of the next product as they lie -- the k slots of an instruction are the keys
//                 {4 h .. 4 h + 3, 8 + 4 h .. 8 + 4 h + 3} of its 16 (h = lane / 32) for both operands
//   O^T += V^T P^T   V stays row-major in LDS; ds_read_b64_tr_b16 hands a lane four keys of its column
// Order of operations as in the composition: s = q k (f32), s * scale, + mask, exp relative to a maximum, sums in f32,
// probabilities rounded to the tensors' type before they meet V (here before the division by their sum, not after).
// The running maximum is only replaced, and the accumulators rescaled, when a score exceeds it by more than 8 (in units
// of log2): p <= 256 loses nothing in either type.
//
// Two forms.  Long rows of queries (NWQ = 4): four wavefronts, 128 rows, share every tile of 64 keys through LDS, two
// tiles in flight, two workgroups a CU.  Few rows
// (NWQ = 1, decode): one block of 32 rows, every wavefront walks tiles of 32 keys of its own -- no barriers, 64 KB of
// keys and values in flight a CU -- and the four partial results meet in LDS.  Queries that share one key / value head
// are rows of one problem (row = query * heads + head).  Where that leaves CUs idle the keys are split over workgroups
// and sdpa_combine_kernel adds the parts.
//
// Bound: for long queries the series of K Q, softmax and P V in a wavefront, behind a wait for all loads and a barrier every
// 64 keys (16 heads, 4096 x 4096, d 128, causal, bf16: the composition 1221 us, of which 729 were the softmax over scores in
// memory, this 91 us = 755 TFLOP/s; the matrix cores and the vector units busy 43 % of the time each, which adds up to the
// 86 % that are not stalls: the two workgroups of a CU hardly run one's softmax under the other's products.  Multiplying the next
// tile's scores among this one's softmax in the wavefront itself was 6 % slower, with and without the order forced.  8 x 8 heads,
// 1918 x 2942, d 64: 4024 -> 119 us); memory for few (8 x 16 heads, one query, 8192 keys: 653 -> 103 us, 5.2 TB/s; a wavefront
// waits 55 %).
// 64 rows is where the forms cross: at 64 rows half of the large form's wavefronts have none.  The form for few rows
// reads every mask buffer element by element (the decode above: 172 us with one).
#include "kernels.hpp"

namespace mi355 {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i2v __attribute__((ext_vector_type(2)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
struct __attribute__((packed, aligned(2))) mask2_t { i2v v; };
struct __attribute__((packed, aligned(4))) mask4_t { f4v v; };
typedef const i4v __attribute__((address_space(3))) *lds_i4_t;
typedef i4v __attribute__((address_space(3))) *lds_w4_t;
typedef s4v __attribute__((address_space(3))) *lds_s4_t;
typedef float __attribute__((address_space(3))) *lds_f_t;

struct sdpa_dev_t {
    mi355_sdpa_desc_t d;
    const char *q, *k, *v;
    char *dst;
    const void *scale, *mask;
    float *part_o, *part_ml; // splits > 1: [split][b * hk][rows][d] and [split][b * hk][rows][2]
    int splits, nq;          // parts of the keys; row blocks
    int rows, hg;            // query rows per key / value head, query heads per key / value head
};

// lane i brings 16 bytes from sbase + voff to LDS byte address lds_addr + 16 i
__device__ __forceinline__ void sdpa_dma16(const void *sbase, unsigned voff, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(sbase)
                 : "memory", "m0");
}

template <int DT>
__device__ __forceinline__ f16v sdpa_mma(i4v a, i4v b, f16v c) {
    if constexpr (DT == MI355_DT_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, a), __builtin_bit_cast(h8v, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ int sdpa_pack(float lo, float hi) {
    if constexpr (DT == MI355_DT_BF16) {
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(int, __builtin_convertvector(f2 {lo, hi}, bf2));
    } else {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(int, h2 {(_Float16)lo, (_Float16)hi});
    }
}

// the same value from the other half of the wavefront, combined
__device__ __forceinline__ float halves_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(f2u(x), f2u(x), false, false);
    return fmaxf(u2f(r[0]), u2f(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(f2u(x), f2u(x), false, false);
    return u2f(r[0]) + u2f(r[1]);
}

// The scale as the composition reads it: in its own type, the reciprocal rounded to that type when inverted.
__device__ __forceinline__ float sdpa_scale(const mi355_sdpa_desc_t &D, const void *p) {
    if (D.scale_dt == MI355_DT_UNDEF) return 1.f;
    float sc = load_float(D.scale_dt, p, 0);
    if (D.invert_scale) {
        const uint32_t bits = cvt_store_bits(D.scale_dt, 1.f / sc);
        sc = D.scale_dt == MI355_DT_F32 ? u2f(bits)
                : D.scale_dt == MI355_DT_BF16 ? u2f(bits << 16) : (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
    }
    return sc;
}

// MASK: 0 no buffer; 1 any buffer, element by element; 2 / 3 a 16-bit / f32 buffer whose keys lie side by side:
// requested ahead of the scores, four keys a load (2 x 16 heads, 1000 x 1500, d 128: 210 us element by element, 62 so)
template <int DT, int D, int MASK, int NWQ>
__global__ void __launch_bounds__(256, 2) sdpa_kernel(const sdpa_dev_t P) {
    constexpr int KT = NWQ == 4 ? 64 : 32;          // keys of a tile
    constexpr int RB = NWQ == 4 ? 128 : 32;         // query rows of a workgroup
    constexpr int ROWB = D * 2;                     // bytes of a row of K or V
    constexpr int TILE = KT * ROWB;                 // bytes of a tile of K or V in LDS
    constexpr int NDMA = TILE / 1024 / NWQ;         // direct-to-LDS loads of a wavefront per tile of K or V
    constexpr int RPD = 1024 / ROWB;                // rows of one such load
    constexpr int QT = D / 16, NT = D / 32, ST = KT / 32;
    constexpr float LOG2E = 1.44269504088896340736f;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const mi355_sdpa_desc_t &Dd = P.d;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l31 = lane & 31, hf = lane >> 5;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;

    // workgroup -> (key / value head, block of rows).  Neighbouring ids take different heads (an XCD then keeps the
    // keys of few heads in its L2).  With a causal mask the blocks differ in length: the long ones first, and when all
    // workgroups are resident at once (two a CU) the second half in the opposite order, so that a CU's two add up alike.
    const int nbh = (int)(Dd.b * Dd.hk);
    const int bh = (int)blockIdx.x % nbh, rank = (int)blockIdx.x / nbh;
    int qb = P.nq - 1 - rank;
    if ((long)P.nq * nbh <= 512 && rank >= (P.nq + 1) / 2) qb = rank - (P.nq + 1) / 2;
    const long bi = bh / Dd.hk, kvh = bh % Dd.hk;
    const int row0 = qb * RB + (NWQ == 4 ? 32 * wave : 0);
    const int row = row0 + l31, rowc = row < P.rows ? row : P.rows - 1;
    const int qi = P.hg == 1 ? rowc : rowc / P.hg;
    const long head = kvh * P.hg + (P.hg == 1 ? 0 : rowc % P.hg);

    // keys this lane's query sees: [0, klim); tiles of the workgroup and of the wavefront
    const int sq = (int)Dd.sq, sk = (int)Dd.sk;
    const int diag = Dd.mask_type == 2 ? 1 : sk - sq + 1;
    auto limit = [&](int q) {
        if (Dd.mask_type < 2) return sk;
        const int e = q + diag;
        return e < 0 ? 0 : (e < sk ? e : sk);
    };
    const int klim = limit(qi);
    auto query_of = [&](int r) { r = r < P.rows ? r : P.rows - 1; return P.hg == 1 ? r : r / P.hg; };
    const int wg_lim = limit(query_of(qb * RB + RB - 1));
    const int w_lo = limit(query_of(row0)), w_hi = limit(query_of(row0 + 31)); // (rows ascend with their limits)
    const int ntiles = (wg_lim + KT - 1) / KT;
    const int per = (ntiles + P.splits - 1) / P.splits;
    const int t_begin = (int)blockIdx.y * per, t_end = t_begin + per < ntiles ? t_begin + per : ntiles;

    float c = sdpa_scale(Dd, P.scale);
    const bool neg = c < 0.f; // folded into Q, so that a larger score stays a larger exponent
    c = neg ? -c : c;
    const float sc = c;
    // (with a buffer the scores stay in units of e until the maximum is taken off: a mask of the type's lowest value
    // times log2(e) would be -inf, and a row of nothing else has to weigh its keys alike)
    constexpr float UNIT = MASK ? LOG2E : 1.f;
    c = MASK ? 1.f : c * LOG2E;
    c = c == 0.f ? 0x1p-149f : c; // (zero must not meet the infinities of masked keys; finite scores times this are 0 to exp2)

    i4v qf[QT];
    {
        const char *qp = P.q + 2 * (bi * Dd.q_stride[0] + head * Dd.q_stride[1] + qi * Dd.q_stride[2]) + 16 * hf;
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            qf[t] = *(const i4v *)(qp + 32 * t);
            if (neg)
#pragma unroll
                for (int e = 0; e < 4; ++e) qf[t][e] ^= (int)0x80008000;
        }
    }
    const char *mrow = MASK ? (const char *)P.mask : nullptr;
    long moff = 0;
    if (MASK) moff = bi * Dd.mask_stride[0] + head * Dd.mask_stride[1] + qi * Dd.mask_stride[2];

    // ---- tiles of K and V: row r, 16-byte chunk ch.  Rows of 256 bytes are whole LDS lines: K's chunks are XOR-ed with
    // the row (32 rows of one chunk are read at a time), V's with the row in steps of 64 bytes (eight rows of 64 bytes
    // are).  Rows of 128 bytes sit two to a line.
    const char *kbase = P.k + 2 * (bi * Dd.k_stride[0] + kvh * Dd.k_stride[1]);
    const char *vbase = P.v + 2 * (bi * Dd.v_stride[0] + kvh * Dd.v_stride[1]);
    const int kpitch = (int)(2 * Dd.k_stride[2]), vpitch = (int)(2 * Dd.v_stride[2]);
    const int dw = NWQ == 4 ? wave * NDMA : 0; // the wavefront's first load of a tile
    const unsigned ring = NWQ == 4 ? 0 : (unsigned)wave * 4 * TILE;
    int drow[NDMA], kch[NDMA], vch[NDMA];
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int s = lane & 15;
        if (D == 128) {
            const int r = (dw + i) * RPD + (lane >> 4);
            drow[i] = r;
            kch[i] = 16 * (s ^ (r & 15));
            vch[i] = 16 * (s ^ ((r & 3) << 2));
        } else {
            const int r = (dw + i) * RPD + 2 * (lane >> 4) + (s >> 3);
            drow[i] = r;
            kch[i] = 16 * ((s & 7) ^ ((r >> 1) & 7));
            vch[i] = 16 * ((s & 7) ^ (4 * ((r >> 1) & 1)));
        }
    }
    auto issue = [&](int t, int buf) __attribute__((always_inline)) {
        const int key0 = t * KT, left = sk - 1 - key0; // rows beyond the last key are fetched from it
        const char *kt = kbase + (long)key0 * kpitch, *vt = vbase + (long)key0 * vpitch;
        const unsigned dst = lds0 + ring + (unsigned)buf * 2 * TILE + (unsigned)dw * 1024;
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int r = drow[i] < left ? drow[i] : left;
            sdpa_dma16(kt, (unsigned)(r * kpitch + kch[i]), dst + (unsigned)i * 1024);
        }
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int r = drow[i] < left ? drow[i] : left;
            sdpa_dma16(vt, (unsigned)(r * vpitch + vch[i]), dst + TILE + (unsigned)i * 1024);
        }
    };
    // fragment addresses inside a tile
    unsigned ka[QT], va[NT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        if (D == 128) ka[t] = (unsigned)(l31 * 256 + (((2 * t + hf) ^ (l31 & 15)) << 4));
        else ka[t] = (unsigned)((l31 >> 1) * 256 + (((l31 & 1) * 8 + ((2 * t + hf) ^ ((l31 >> 1) & 7))) << 4));
    }
    {
        const int li = lane & 15, g = lane >> 4, r = 4 * hf + (li >> 2); // key row of the lane's 8 bytes
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int ch = 4 * n + 2 * (g & 1) + ((li & 3) >> 1);
            if (D == 128) va[n] = (unsigned)(r * 256 + ((ch ^ ((r & 3) << 2)) << 4) + 8 * (li & 1));
            else va[n] = (unsigned)((r >> 1) * 256 + (((r & 1) * 8 + (ch ^ (4 * ((r >> 1) & 1)))) << 4) + 8 * (li & 1));
        }
    }

    // Rows beyond the last key hold that key's values again, and meet probabilities of 0: zeros instead, since an
    // infinity there would make NaN of a result that is infinite.  (A row of V fills its ROWB bytes of the tile.)
    auto clear_tail = [&](int t, int buf, int first, int step) __attribute__((always_inline)) {
        const unsigned v0 = lds0 + ring + (unsigned)buf * 2 * TILE + TILE;
        for (int at = (sk - t * KT) * ROWB + 16 * first; at < TILE; at += 16 * step)
            *(lds_w4_t)(size_t)(v0 + (unsigned)at) = i4v {0, 0, 0, 0};
    };

    f16v o[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[n][r] = 0.f;
    float m = -INFINITY, l = 0.f; // running maximum (in units of 1 / UNIT of log2), this lane half's sum of p

    auto tile = [&](int t, int buf) __attribute__((always_inline)) {
        const unsigned kl = lds0 + ring + (unsigned)buf * 2 * TILE, vl = kl + TILE;
        const int key0 = t * KT;
        f16v s[ST];
#pragma unroll
        for (int x = 0; x < ST; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[x][r] = 0.f;
        i2v m2[ST * 4];
        f4v m4[ST * 4];
        if (MASK >= 2) {
#pragma unroll
            for (int x = 0; x < ST; ++x)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    // (rows start at any element: loads of the element's alignment; the last, partial tile one by one)
                    const int key = key0 + 32 * x + 8 * a + 4 * hf;
                    if (key0 + KT <= sk) {
                        if (MASK == 2) m2[4 * x + a] = ((const mask2_t *)(mrow + 2 * (moff + key)))->v;
                        else m4[4 * x + a] = ((const mask4_t *)(mrow + 4 * (moff + key)))->v;
                    } else {
                        uint32_t w[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const long at = moff + (key + e < sk ? key + e : sk - 1);
                            w[e] = MASK == 2 ? ((const uint16_t *)mrow)[at] : ((const uint32_t *)mrow)[at];
                        }
                        if (MASK == 2) m2[4 * x + a] = i2v {(int)(w[0] | w[1] << 16), (int)(w[2] | w[3] << 16)};
                        else m4[4 * x + a] = f4v {u2f(w[0]), u2f(w[1]), u2f(w[2]), u2f(w[3])};
                    }
                }
        }
#pragma unroll
        for (int d = 0; d < QT; ++d)
#pragma unroll
            for (int x = 0; x < ST; ++x)
                s[x] = sdpa_mma<DT>(*(lds_i4_t)(size_t)(kl + ka[d] + x * 32 * ROWB), qf[d], s[x]);
        if (MASK == 2) {
            const bool bf = Dd.mask_dt == MI355_DT_BF16;
#pragma unroll
            for (int x = 0; x < ST; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t w = (uint32_t)m2[4 * x + r / 4][(r % 4) / 2];
                    const float add = bf ? u2f((r & 1) ? w & 0xffff0000u : w << 16)
                                         : (float)__builtin_bit_cast(_Float16, (unsigned short)((r & 1) ? w >> 16 : w));
                    s[x][r] = s[x][r] * sc + add;
                }
        } else if (MASK == 3) {
#pragma unroll
            for (int x = 0; x < ST; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[x][r] = s[x][r] * sc + m4[4 * x + r / 4][r % 4];
        } else if (MASK == 1) {
#pragma unroll
            for (int x = 0; x < ST; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int key = key0 + 32 * x + 8 * (r / 4) + 4 * hf + r % 4;
                    key = key < sk ? key : sk - 1;
                    s[x][r] = s[x][r] * sc + load_float(Dd.mask_dt, mrow, moff + key * Dd.mask_stride[3]);
                }
        }
        if (key0 + KT > w_lo) { // some lane's limit lies inside the tile
#pragma unroll
            for (int x = 0; x < ST; ++x)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (key0 + 32 * x + 8 * (r / 4) + 4 * hf + r % 4 >= klim) s[x][r] = -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int x = 0; x < ST; ++x)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[x][r]);
        mx = halves_max(mx) * c;
        if (__builtin_amdgcn_ballot_w64(mx > m + 8.f / UNIT) != 0) {
            const float mn = fmaxf(m, mx);
            const float f = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m - mn) * UNIT);
            m = mn;
            l *= f;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[n][r] *= f;
        }
        const float shift = m == -INFINITY ? 0.f : m; // a row of -inf so far: exp2(-inf), not exp2(-inf + inf)
        i4v p[KT / 16];
        float sum = 0.f;
#pragma unroll
        for (int x = 0; x < ST; ++x)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float p0 = __builtin_amdgcn_exp2f(MASK ? (s[x][r] - shift) * UNIT : __builtin_fmaf(s[x][r], c, -shift));
                const float p1 = __builtin_amdgcn_exp2f(MASK ? (s[x][r + 1] - shift) * UNIT : __builtin_fmaf(s[x][r + 1], c, -shift));
                sum += p0 + p1;
                p[2 * x + r / 8][(r % 8) / 2] = sdpa_pack<DT>(p0, p1);
            }
        l += sum;
#pragma unroll
        for (int ks = 0; ks < KT / 16; ++ks)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const unsigned at = vl + va[n] + (unsigned)ks * 16 * ROWB;
                const i2v lo = __builtin_bit_cast(i2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(size_t)at));
                const i2v hi = __builtin_bit_cast(i2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(size_t)(at + 8 * ROWB)));
                o[n] = sdpa_mma<DT>(i4v {lo[0], lo[1], hi[0], hi[1]}, p[ks], o[n]);
            }
    };

    if constexpr (NWQ == 4) {
        if (t_begin < t_end) issue(t_begin, 0);
        for (int t = t_begin; t < t_end; ++t) {
            const int buf = (t - t_begin) & 1;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads(); // the tile is in LDS, and everybody is done with the other buffer
            if (t + 1 < t_end) issue(t + 1, buf ^ 1);
            if (t * KT + KT > sk) { // the last tile, partly filled
                clear_tail(t, buf, (int)threadIdx.x, 256);
                __syncthreads();
            }
            if (t * KT < w_hi) tile(t, buf); // (a tile beyond this wavefront's diagonal holds nothing for it)
        }
    } else {
        int buf = 0;
        if (t_begin + wave < t_end) issue(t_begin + wave, 0);
        for (int t = t_begin + wave; t < t_end; t += 4) {
            const bool more = t + 4 < t_end;
            if (more) {
                // the other buffer was read in the previous iteration: those reads are back before the loads overwrite it
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                issue(t + 4, buf ^ 1);
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NDMA) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            if (t * KT + KT > sk) clear_tail(t, buf, lane, 64); // (a wavefront's own tile: its LDS accesses keep their order)
            tile(t, buf);
            buf ^= 1;
        }
    }
    l = halves_sum(l);

    int n0 = 0; // the first 32-column block of dst that this wavefront finishes (NWQ = 1: the only one)
    if constexpr (NWQ == 1) {
        // four partial results of the same rows: [wave][block][register][lane], then m and l
        __syncthreads();
        const unsigned mine = lds0 + (unsigned)wave * (NT * 16 * 256);
        const unsigned ml = lds0 + 4 * (NT * 16 * 256);
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) *(lds_f_t)(size_t)(mine + (unsigned)((n * 16 + r) * 64 + lane) * 4) = o[n][r];
        *(lds_f_t)(size_t)(ml + (unsigned)(wave * 128 + lane) * 4) = m;
        *(lds_f_t)(size_t)(ml + (unsigned)(wave * 128 + 64 + lane) * 4) = l;
        __syncthreads();
        float mw[4], mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            mw[w] = *(lds_f_t)(size_t)(ml + (unsigned)(w * 128 + lane) * 4);
            mm = fmaxf(mm, mw[w]);
        }
        float f[4];
        l = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            f[w] = mm == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((mw[w] - mm) * UNIT);
            l += f[w] * *(lds_f_t)(size_t)(ml + (unsigned)(w * 128 + 64 + lane) * 4);
        }
        m = mm;
        // wavefront w takes block w (the upper two have none when there are two)
        n0 = wave < NT ? wave : NT;
        if (n0 < NT) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    v += f[w] * *(lds_f_t)(size_t)(lds0 + (unsigned)(((w * NT + n0) * 16 + r) * 64 + lane) * 4);
                o[0][r] = v;
            }
        }
    }
    if (row >= P.rows) return;
    if (P.splits > 1) {
        const long at = ((long)blockIdx.y * nbh + bh) * P.rows + row;
        if (n0 == 0 && hf == 0) {
            P.part_ml[2 * at] = m;
            P.part_ml[2 * at + 1] = l;
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if (NWQ == 1 && n != 0) break;
            if (NWQ == 1 && n0 >= NT) break;
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *(f4v *)(P.part_o + at * D + 32 * (NWQ == 1 ? n0 : n) + 8 * a + 4 * hf)
                        = f4v {o[n][4 * a], o[n][4 * a + 1], o[n][4 * a + 2], o[n][4 * a + 3]};
        }
        return;
    }
    float inv = 1.f / l; // 0 / 0 = NaN for a fully masked row, as in the composition
    if (Dd.inf_as_zero && l == 0.f) inv = 0.f;
    const long doff = bi * Dd.dst_stride[0] + head * Dd.dst_stride[1] + qi * Dd.dst_stride[2];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        if (NWQ == 1 && n != 0) break;
        if (NWQ == 1 && n0 >= NT) break;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const long at = doff + 32 * (NWQ == 1 ? n0 : n) + 8 * a + 4 * hf;
            const float v0 = o[n][4 * a] * inv, v1 = o[n][4 * a + 1] * inv, v2 = o[n][4 * a + 2] * inv, v3 = o[n][4 * a + 3] * inv;
            if (Dd.dst_dt == MI355_DT_F32) *(f4v *)((float *)P.dst + at) = f4v {v0, v1, v2, v3};
            else if (Dd.dst_dt == MI355_DT_BF16)
                *(i2v *)((uint16_t *)P.dst + at) = i2v {sdpa_pack<MI355_DT_BF16>(v0, v1), sdpa_pack<MI355_DT_BF16>(v2, v3)};
            else *(i2v *)((uint16_t *)P.dst + at) = i2v {sdpa_pack<MI355_DT_F16>(v0, v1), sdpa_pack<MI355_DT_F16>(v2, v3)};
        }
    }
}

// The parts of the keys added up: D / 4 lanes a row, four columns each.
__global__ void __launch_bounds__(256) sdpa_combine_kernel(const sdpa_dev_t P) {
    const mi355_sdpa_desc_t &Dd = P.d;
    const int tpr = (int)Dd.d / 4;
    const long nbh = Dd.b * Dd.hk, id = (long)blockIdx.x * (256 / tpr) + threadIdx.x / tpr;
    if (id >= nbh * P.rows) return;
    const int col = 4 * (threadIdx.x % tpr);
    const long total = nbh * P.rows;
    const float unit = Dd.mask_type == 1 ? 1.44269504088896340736f : 1.f; // as in sdpa_kernel
    float mm = -INFINITY;
    for (int s = 0; s < P.splits; ++s) mm = fmaxf(mm, P.part_ml[2 * (s * total + id)]);
    float l = 0.f;
    f4v acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < P.splits; ++s) {
        const long at = s * total + id;
        const float f = mm == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((P.part_ml[2 * at] - mm) * unit);
        l += f * P.part_ml[2 * at + 1];
        const f4v v = *(const f4v *)(P.part_o + at * Dd.d + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += f * v[e];
    }
    float inv = 1.f / l;
    if (Dd.inf_as_zero && l == 0.f) inv = 0.f;
    const long bh = id / P.rows, row = id % P.rows;
    const long bi = bh / Dd.hk, kvh = bh % Dd.hk, qi = row / P.hg, head = kvh * P.hg + row % P.hg;
    const long at = bi * Dd.dst_stride[0] + head * Dd.dst_stride[1] + qi * Dd.dst_stride[2] + col;
    const float v0 = acc[0] * inv, v1 = acc[1] * inv, v2 = acc[2] * inv, v3 = acc[3] * inv;
    if (Dd.dst_dt == MI355_DT_F32) *(f4v *)((float *)P.dst + at) = f4v {v0, v1, v2, v3};
    else if (Dd.dst_dt == MI355_DT_BF16)
        *(i2v *)((uint16_t *)P.dst + at) = i2v {sdpa_pack<MI355_DT_BF16>(v0, v1), sdpa_pack<MI355_DT_BF16>(v2, v3)};
    else *(i2v *)((uint16_t *)P.dst + at) = i2v {sdpa_pack<MI355_DT_F16>(v0, v1), sdpa_pack<MI355_DT_F16>(v2, v3)};
}

struct sdpa_plan_t {
    bool few;     // the form for few rows of queries
    int nq, splits;
    long rows;
    size_t part_o, total;
};

sdpa_plan_t sdpa_plan(const mi355_sdpa_desc_t &d) {
    sdpa_plan_t p;
    p.rows = d.h / d.hk * d.sq;
    p.few = p.rows <= 64;
    const int rb = p.few ? 32 : 128, kt = p.few ? 32 : 64;
    p.nq = (int)((p.rows + rb - 1) / rb);
    // Split the keys while workgroups are fewer than the device holds (one or two a CU) and every part still has a
    // few tiles for each of its wavefronts
    const long wgs = (long)p.nq * d.b * d.hk, tiles = (d.sk + kt - 1) / kt, least = p.few ? 8 : 4;
    long s = wgs >= 256 ? 1 : 512 / wgs;
    if (s > tiles / least) s = tiles / least;
    if (s < 1) s = 1;
    p.splits = (int)s;
    p.part_o = s > 1 ? (size_t)s * d.b * d.hk * p.rows * d.d * 4 : 0;
    p.total = s > 1 ? p.part_o + (size_t)s * d.b * d.hk * p.rows * 8 : 0;
    return p;
}

template <int DT, int D, int MASK, int NWQ>
int sdpa_go(const sdpa_dev_t &P, unsigned wgs, hipStream_t stream) {
    constexpr int KT = NWQ == 4 ? 64 : 32;
    constexpr int RING = (NWQ == 4 ? 1 : 4) * 4 * KT * D * 2, MEET = 4 * (D / 32 * 16 * 256) + 4 * 512;
    constexpr int LDS = NWQ == 1 && MEET > RING ? MEET : RING;
    if (const int st = ensure_dynamic_lds((const void *)sdpa_kernel<DT, D, MASK, NWQ>, LDS, "sdpa")) return st;
    hipLaunchKernelGGL((sdpa_kernel<DT, D, MASK, NWQ>), dim3(wgs, (unsigned)P.splits), dim3(256), LDS, stream, P);
    return MI355_SUCCESS;
}

template <int DT, int D>
int sdpa_pick(const sdpa_dev_t &P, bool few, unsigned wgs, hipStream_t stream) {
    if (P.d.mask_type != 1) return few ? sdpa_go<DT, D, 0, 1>(P, wgs, stream) : sdpa_go<DT, D, 0, 4>(P, wgs, stream);
    if (few) return sdpa_go<DT, D, 1, 1>(P, wgs, stream);
    if (P.d.mask_stride[3] != 1) return sdpa_go<DT, D, 1, 4>(P, wgs, stream);
    return P.d.mask_dt == MI355_DT_F32 ? sdpa_go<DT, D, 3, 4>(P, wgs, stream) : sdpa_go<DT, D, 2, 4>(P, wgs, stream);
}

} // namespace
} // namespace mi355

using namespace mi355;

extern "C" int mi355_sdpa_query(const mi355_sdpa_desc_t *d, size_t *scratch_bytes) {
    if (!d || !scratch_bytes) return MI355_INVALID_ARGUMENTS;
    *scratch_bytes = 0;
    auto fp = [](int dt) { return dt == MI355_DT_F32 || dt == MI355_DT_BF16 || dt == MI355_DT_F16; };
    if (d->dt != MI355_DT_BF16 && d->dt != MI355_DT_F16) return MI355_UNIMPLEMENTED;
    if (!fp(d->dst_dt) || (d->d != 64 && d->d != 128)) return MI355_UNIMPLEMENTED;
    if (d->b < 1 || d->h < 1 || d->hk < 1 || d->sq < 1 || d->sk < 1 || (d->hk != 1 && d->hk != d->h)) return MI355_UNIMPLEMENTED;
    if (d->scale_dt != MI355_DT_UNDEF && !fp(d->scale_dt)) return MI355_UNIMPLEMENTED;
    if (d->mask_type < 0 || d->mask_type > 3 || (d->mask_type == 1 && !fp(d->mask_dt))) return MI355_UNIMPLEMENTED;
    // 16-byte loads of rows at 32-bit offsets inside a tile; 8- or 16-byte stores of dst
    for (const int64_t *s : {d->q_stride, d->k_stride, d->v_stride})
        for (int i = 0; i < 3; ++i)
            if (s[i] % 8 != 0 || s[i] < 0) return MI355_UNIMPLEMENTED;
    for (int i = 0; i < 3; ++i)
        if (d->dst_stride[i] % 4 != 0 || d->dst_stride[i] < 0) return MI355_UNIMPLEMENTED;
    if (d->k_stride[2] >= (1L << 23) || d->v_stride[2] >= (1L << 23)) return MI355_UNIMPLEMENTED;
    const long rows = d->h / d->hk * d->sq;
    if (rows >= (1L << 30) || d->sk >= (1L << 30) || d->sq >= (1L << 30)) return MI355_UNIMPLEMENTED;
    const sdpa_plan_t p = sdpa_plan(*d);
    if ((long)p.nq * d->b * d->hk >= (1L << 31)) return MI355_UNIMPLEMENTED;
    *scratch_bytes = p.total;
    return MI355_SUCCESS;
}

extern "C" int mi355_sdpa_launch(const mi355_sdpa_desc_t *d, const void *q, const void *k, const void *v, void *dst,
        const void *scale, const void *mask, void *scratch, void *stream) {
    size_t need = 0;
    const int st = mi355_sdpa_query(d, &need);
    if (st != MI355_SUCCESS) return st;
    if (!q || !k || !v || !dst || (d->scale_dt != MI355_DT_UNDEF && !scale) || (d->mask_type == 1 && !mask) || (need && !scratch)) {
        set_error("sdpa: a tensor or %zu bytes of scratch are missing", need);
        return MI355_INVALID_ARGUMENTS;
    }
    if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dst) & 15) != 0) {
        set_error("sdpa: queries, keys, values and dst must be 16-byte aligned");
        return MI355_UNIMPLEMENTED;
    }
    const sdpa_plan_t p = sdpa_plan(*d);
    sdpa_dev_t P {};
    P.d = *d;
    P.q = (const char *)q;
    P.k = (const char *)k;
    P.v = (const char *)v;
    P.dst = (char *)dst;
    P.scale = scale;
    P.mask = mask;
    P.part_o = (float *)scratch;
    P.part_ml = (float *)((char *)scratch + p.part_o);
    P.splits = p.splits;
    P.nq = p.nq;
    P.rows = (int)p.rows;
    P.hg = (int)(d->h / d->hk);
    const unsigned wgs = (unsigned)(p.nq * d->b * d->hk);
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (d->dt == MI355_DT_BF16) rc = d->d == 128 ? sdpa_pick<MI355_DT_BF16, 128>(P, p.few, wgs, s) : sdpa_pick<MI355_DT_BF16, 64>(P, p.few, wgs, s);
    else rc = d->d == 128 ? sdpa_pick<MI355_DT_F16, 128>(P, p.few, wgs, s) : sdpa_pick<MI355_DT_F16, 64>(P, p.few, wgs, s);
    if (rc != MI355_SUCCESS) return rc;
    if (p.splits > 1) {
        const long rpb = 256 / (d->d / 4), total = d->b * d->hk * p.rows;
        hipLaunchKernelGGL(sdpa_combine_kernel, dim3((unsigned)((total + rpb - 1) / rpb)), dim3(256), 0, s, P);
    }
    return hipGetLastError() == hipSuccess ? MI355_SUCCESS : MI355_RUNTIME_ERROR;
}
