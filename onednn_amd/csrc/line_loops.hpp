// The K loops of the tiles that read whole 128-byte lines: int8, fp8, MXFP8, MXFP4 and the 16-bit types.
//
// A step is 128 bytes of K of every row, so that a wavefront's direct-to-LDS load brings 8 whole lines.  The loops
// before these took 64 bytes a step: a load then touches 16 half lines, the L2 is asked twice for every line, and the
// loads hold their wavefronts and burn the power budget of the matrix cores.  Same tiles, same MFMAs, 8192^3 on one
// device, 64-byte steps against these: bf16 0.81 -> 0.72 ms, int8 0.47 -> 0.37; matrix cores busy 0.64 -> 0.82 of the
// cycles at an unchanged 1.75-1.8 GHz.
//
// The LDS ring holds two steps (A: 256 rows, B^T: BN rows, 128 bytes each).  What makes two enough is that a step is
// released in four parts: the rows and columns of a wavefront's part are halved, a step's products are taken as four
// quadrants (64 rows x half of the columns), and the part of the ring that holds a half is loaded again, for two
// steps on, as soon as every wavefront has that half in registers: loads lead their use by 1.5 to 1.75 steps.
//
// LDS rows are 128 bytes, the eight 16-byte chunks XOR-swizzled by bits 1-3 of the row (on the global side of the
// load), which keeps the fragment reads -- 16 rows x 4 chunks -- free of bank conflicts (SQ_LDS_BANK_CONFLICT = 0).
//
// Fragments: 16 rows x 128 bytes, two 16-byte chunks a lane (row lane % 16, chunks lane / 16 and 4 + lane / 16).  An
// instruction of 64 bytes of K (bf16 / f16 16x16x32, int8 16x16x64, fp4 16x16x128) takes one of them, two a pair; fp8
// 16x16x128 takes both.
//
// An operand of the 16-bit types may also lie the other way round, its rows (of src) or columns (of the weights)
// contiguous and K across them: what a transposed layer has, backward by data in its weights and backward by weights in
// both operands.  Its part of a step is 64 k of whole 512- or 256-byte lines, halved by k (32 each) where the other kind is
// halved by rows; a fragment comes out of LDS through ds_read_b64_tr_b16, which hands lane (r, q) the four k of its row
// from four lines, and is then the same as the other kind's.  Copying such operands K-contiguous first took 144 of the
// 735 us of a training step (2048 x 14336 x 4096).  The 32-byte units of a line are XOR-swizzled by bits 0, 1 and 3 of k:
// the eight lines that half a wavefront reads 32 bytes of start at one bank.
//
// A last step that K does not fill (any whole number of 16-byte chunks, any K where both operands lie the other way
// round) loads no chunk beyond the row's end -- the
// lanes of those chunks repeat the last one -- and they are zeroed in the fragments of both operands (both, so that no
// Inf or NaN meets a zero).
#pragma once
#include "gemm_core.hpp"

namespace mi355 {
namespace gemm {

constexpr int LKB = 128; // bytes of K per row and step

__device__ __forceinline__ int line_swz(int row) { return (row >> 1) & 7; }

// operands whose rows / columns are contiguous instead of K
template <class Mma, class = void>
struct line_form {
    static constexpr bool AKM = false, BKM = false;
};
template <class Mma>
struct line_form<Mma, std::enable_if_t<(Mma::A_KM || Mma::B_KM)>> {
    static constexpr bool AKM = Mma::A_KM, BKM = Mma::B_KM;
};
// the swizzle of a line of such an operand, in 32-byte units
__device__ __forceinline__ int kline_swz(int k) { return (k & 3) | ((k >> 3) & 1) << 2; }

typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef v4s_t __attribute__((address_space(3))) *lds_v4s_ptr_t;
typedef int v2i_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2i_t lds_read_tr16(unsigned addr) {
    return __builtin_bit_cast(v2i_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_ptr_t)(size_t)addr));
}

struct line_pair_t {
    v4i c[2];
    __device__ __forceinline__ v8i whole() const {
        return v8i {c[0][0], c[0][1], c[0][2], c[0][3], c[1][0], c[1][1], c[1][2], c[1][3]};
    }
};

template <class G>
struct line_geo_t {
    static constexpr int NW = G::NW, BN = G::BN, WC = G::WCOLS;
    static constexpr int QC = WC / 32;                   // 16-column tiles in a half of a wavefront's columns
    static constexpr int STAGE_BYTES = (BM + BN) * LKB;  // 64 KB, or 48 KB of the 256 x 128 tile
    static constexpr int RING_BYTES = 2 * STAGE_BYTES;
    static constexpr int B_OFF = BM * LKB;
    static constexpr int DPA = 16 / NW;                  // loads per wavefront of a half of the A rows, of the B^T rows
    static constexpr int DPB = DPA * BN / 256;
    // the epilogue's 16 KB per wavefront
    static_assert(RING_BYTES >= NW * 16384, "epilogue LDS");
};

// e8m0 scales per 32 k of both operands, in the order that mx_scales_rows_kernel / mx_scales_blocks_kernel
// (kern_mxf4.hip) write: per four blocks of k and group of 64 rows 64 dwords, dword 4 r + q = the bytes of block q of rows
// r, 16 + r, 32 + r, 48 + r.  Lane (r, q) of an instruction's operands reads one dword and has the scales of four
// fragments, which the instruction picks by its op_sel bits.
struct line_scales_t {
    const char *a, *b;     // of the tile's first row and column, step 0
    long a_pitch, b_pitch; // bytes between sets of four blocks
    int sets;              // sets of K
};

struct line_scales_args_t { // of a problem
    const char *a, *b;
    long a_bs, b_bs, a_pitch, b_pitch;
    int sets;
    __host__ __device__ __forceinline__ line_scales_t tile(long batch, long m0, long n0) const {
        return line_scales_t {a + batch * a_bs + m0 * 4, b + batch * b_bs + n0 * 4, a_pitch, b_pitch, sets};
    }
};

// Loads of one workgroup: every wavefront's addresses, the ring, the scales' ring behind it.
template <class Mma>
struct line_loader_t {
    using G = typename Mma::G;
    using L = line_geo_t<G>;
    static constexpr int NS = Mma::SCALE_SETS;                  // sets of four blocks in a step
    static constexpr int SG = 4 + G::BN / 64;                   // groups of 64 rows in a set, A's first
    static constexpr int SCALE_BYTES = NS * SG * 256;           // of a step
    static constexpr int EX = (NS * SG + G::NW - 1) / G::NW;    // scale loads per wavefront and step
    static constexpr int LDS_BYTES = L::RING_BYTES + 2 * SCALE_BYTES;

    static constexpr bool AKM = line_form<Mma>::AKM, BKM = line_form<Mma>::BKM;
    static constexpr int ARB = 2 * BM, BRB = 2 * G::BN; // bytes of a line of 64 k's operand part

    unsigned lds0;
    const char *a_tile, *b_tile;
    int nst, lane, wave, krows;
    long lda, ldb;
    unsigned tail_mask;          // all ones if the last step is partial
    unsigned va[2][L::DPA], vb[2][L::DPB], over[2];
    unsigned la[2][L::DPA], lb[2][L::DPB]; // uniform
    const char *sbase[EX ? EX : 1];
    long spitch[EX ? EX : 1];
    int sset[EX ? EX : 1], sets;
    unsigned sdst[EX ? EX : 1];

    // row (of 32) that instruction i of this wavefront brings to this lane, lines of RB bytes
    template <int RB, int D>
    __device__ __forceinline__ int krow(int i) const {
        return (wave * D + i) * (1024 / RB) + lane / (RB / 16);
    }
    template <int RB, int D>
    __device__ __forceinline__ unsigned kvoff(int i, long ld, long left) const {
        const int r = krow<RB, D>(i), chunk = (lane & (RB / 16 - 1)) ^ (kline_swz(r) << 1);
        return (unsigned)(r * ld + min((long)chunk, left / 8 - 1) * 16); // (columns beyond the last: it again)
    }
    __device__ __forceinline__ void init(char *smem, const char *a_, const char *b_, long lda_, long ldb_, long rows_a_left,
            long rows_b_left, long kbytes, const line_scales_t &sc) {
        lda = lda_;
        ldb = ldb_;
        krows = scalar_int((int)(kbytes / 2));
        lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;
        a_tile = scalar_ptr(a_);
        b_tile = scalar_ptr(b_);
        const int rem = (int)(kbytes % LKB + 15) / 16; // chunks of a partial last step
        nst = scalar_int((int)(kbytes / LKB) + (rem ? 1 : 0));
        tail_mask = (unsigned)scalar_int(rem ? -1 : 0);
        const int t = threadIdx.x;
        lane = t & 63;
        wave = __builtin_amdgcn_readfirstlane(t >> 6);
        const int r8 = lane >> 3;
        // a load is 8 rows: which of the two parities of row block decides the swizzle
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int c = (lane & 7) ^ line_swz(par * 8 + r8);
            over[par] = (unsigned)((c - min(c, rem - 1)) * 16); // back to the last whole chunk
            if (rem == 0) over[par] = 0;
        }
        constexpr int BPW = L::WC / 16; // row blocks of a half of a wavefront's columns
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < L::DPA; ++i) {
                if constexpr (AKM) {
                    va[h][i] = kvoff<ARB, L::DPA>(i, lda, rows_a_left);
                    la[h][i] = (unsigned)(h * 32 * ARB + (wave * L::DPA + i) * 1024);
                    continue;
                }
                const int j = wave * L::DPA + i, row0 = (j / 8) * 128 + h * 64 + (j % 8) * 8;
                const int c = (lane & 7) ^ line_swz(row0 + r8);
                const long r = min((long)(row0 + r8), rows_a_left - 1);
                va[h][i] = (unsigned)(r * lda + c * 16);
                la[h][i] = (unsigned)(row0 * LKB);
            }
#pragma unroll
            for (int i = 0; i < L::DPB; ++i) {
                if constexpr (BKM) {
                    vb[h][i] = kvoff<BRB, L::DPB>(i, ldb, rows_b_left);
                    lb[h][i] = (unsigned)(L::B_OFF + h * 32 * BRB + (wave * L::DPB + i) * 1024);
                    continue;
                }
                const int j = wave * L::DPB + i, row0 = (j / BPW) * L::WC + h * (L::WC / 2) + (j % BPW) * 8;
                const int c = (lane & 7) ^ line_swz(row0 + r8);
                const long r = min((long)(row0 + r8), rows_b_left - 1);
                vb[h][i] = (unsigned)(r * ldb + c * 16);
                lb[h][i] = (unsigned)(L::B_OFF + row0 * LKB);
            }
        }
        if constexpr (NS > 0) {
            sets = scalar_int(sc.sets);
#pragma unroll
            for (int k = 0; k < EX; ++k) {
                // (every wavefront issues the same number of loads: the surplus ones bring the last group again)
                const int e = min(wave * EX + k, NS * SG - 1), u = e / SG, g = e % SG;
                const bool of_a = g < 4;
                spitch[k] = of_a ? sc.a_pitch : sc.b_pitch;
                sbase[k] = scalar_ptr(of_a ? sc.a + g * 256 : sc.b + (g - 4) * 256);
                sset[k] = u;
                sdst[k] = (unsigned)(L::RING_BYTES + e * 256);
            }
        }
    }
    // Steps from 0 on that load and multiply whole steps inside K only (a step loads two ahead); the rest are END
    // steps: loads past the last step are issued all the same, clamped to the last one and into a slot nobody reads
    // again -- one outstanding-load count fits every step -- and a partial last step is taken care of.
    __device__ __forceinline__ int steady() const { return nst - (tail_mask ? 3 : 2); }
    __device__ __forceinline__ int clamp(int s) const { return s < nst ? s : nst - 1; }
    // instruction i of half h (32 k) of a step's part of an operand whose lines run across K; lines beyond K: the last one
    template <bool END, int RB, int D>
    __device__ __forceinline__ void load_k1(const char *tile, long ld, unsigned voff, int h, int i, int sc, unsigned dst) const {
        if (END) {
            const int r = krow<RB, D>(i), row = min(h * 32 + r, krows - 1 - sc * 64);
            dma16(tile + (long)sc * 64 * ld, voff + (unsigned)((row - r) * (int)ld), dst);
        } else {
            dma16(tile + ((long)sc * 64 + h * 32) * ld, voff, dst);
        }
    }
    template <bool END>
    __device__ __forceinline__ void load_a1(int h, int i, int s, int slot) const {
        const int sc = END ? clamp(s) : s;
        if constexpr (AKM) {
            load_k1<END, ARB, L::DPA>(a_tile, lda, va[h][i], h, i, sc, lds0 + slot * L::STAGE_BYTES + la[h][i]);
            return;
        }
        const unsigned back = END ? over[block_parity(L::DPA, i)] & (sc == nst - 1 ? tail_mask : 0u) : 0u;
        dma16(a_tile + (long)sc * LKB, va[h][i] - back, lds0 + slot * L::STAGE_BYTES + la[h][i]);
    }
    template <bool END>
    __device__ __forceinline__ void load_b1(int h, int i, int s, int slot) const {
        const int sc = END ? clamp(s) : s;
        if constexpr (BKM) {
            load_k1<END, BRB, L::DPB>(b_tile, ldb, vb[h][i], h, i, sc, lds0 + slot * L::STAGE_BYTES + lb[h][i]);
            return;
        }
        const unsigned back = END ? over[block_parity(L::DPB, i)] & (sc == nst - 1 ? tail_mask : 0u) : 0u;
        dma16(b_tile + (long)sc * LKB, vb[h][i] - back, lds0 + slot * L::STAGE_BYTES + lb[h][i]);
    }
    // a wavefront's blocks of 8 rows start at an even one
    static __device__ __forceinline__ constexpr int block_parity(int per_wave, int i) {
        return per_wave % 2 == 0 ? i & 1 : 0;
    }
    template <bool END>
    __device__ __forceinline__ void load_a(int h, int s, int slot) const {
#pragma unroll
        for (int i = 0; i < L::DPA; ++i) load_a1<END>(h, i, s, slot);
    }
    template <bool END>
    __device__ __forceinline__ void load_b(int h, int s, int slot) const {
        static_assert(L::DPA % 2 == 0 && L::DPB % 2 == 0, "block parity");
#pragma unroll
        for (int i = 0; i < L::DPB; ++i) load_b1<END>(h, i, s, slot);
    }
    template <bool END>
    __device__ __forceinline__ void load_scales(int s, int slot) const {
        if constexpr (NS > 0) {
#pragma unroll
            for (int k = 0; k < EX; ++k)
                // (a second set that K does not reach: the last one again, its products are with zeroed fragments)
                dma4(sbase[k] + (long)(END ? min(clamp(s) * NS + sset[k], sets - 1) : s * NS + sset[k]) * spitch[k], (unsigned)lane * 4u, lds0 + sdst[k] + slot * SCALE_BYTES);
        }
    }
};

// A wavefront's fragments: both halves of its rows (four 16-row tiles each) and of its columns.
template <class Mma>
struct line_frags_t {
    using G = typename Mma::G;
    using L = line_geo_t<G>;
    using Ld = line_loader_t<Mma>;
    static constexpr int QC = L::QC, NS = Ld::NS;
    line_pair_t a[2][4], b[2][QC];
    int sa[2][NS ? NS : 1], sb[2][NS ? NS : 1]; // sb: of this step and, read ahead, of the next
    // LDS addresses of chunk u of fragment 0 by slot (the fragments' offsets ride in the read's offset field, which does
    // not reach from one slot to the other), and of the lane's scale dword
    unsigned ra[2][2], rb[2][2], rs;
    int inside[2]; // bytes of this lane's chunk u that lie inside K in a partial last step
    // the other kind of operand: this lane's address inside a slot, but for the tile (XOR of its 32-byte unit), the lines
    // of 4 further k and the half
    unsigned ka, kb, slot0;

    __device__ __forceinline__ void init(const Ld &ld, long kbytes) {
        const int t = threadIdx.x, lane = t & 63, r = lane & 15, q = lane >> 4;
        const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = G::wm(wave), wn = G::wn(wave);
        const int rem = (int)(kbytes % LKB), i4 = (lane & 15) >> 2, g = i4 | (q & 1) << 2;
        slot0 = ld.lds0;
        ka = (unsigned)((8 * q + i4) * Ld::ARB + ((wm * 8 ^ g) << 5) + (lane & 3) * 8);
        kb = (unsigned)((8 * q + i4) * Ld::BRB + ((wn * (L::WC / 16) ^ g) << 5) + (lane & 3) * 8);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const unsigned c = (unsigned)(((u * 4 + q) ^ line_swz(r)) << 4);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                ra[s][u] = ld.lds0 + s * L::STAGE_BYTES + (wm * 128 + r) * LKB + c;
                rb[s][u] = ld.lds0 + s * L::STAGE_BYTES + L::B_OFF + (wn * L::WC + r) * LKB + c;
            }
            inside[u] = min(max(rem - (u * 4 + q) * 16, 0), 16);
        }
        rs = ld.lds0 + L::RING_BYTES + (r * 4 + q) * 4;
        if constexpr (NS == 0) sa[0][0] = sa[1][0] = sb[0][0] = sb[1][0] = 0;
    }
    // MXFP4's last steps (END), where the slot is not a constant, work the address out from one: its two sets of scales
    // leave the eight-wavefront loop no registers, and the general epilogue's kernel kept 22 in scratch memory, whose
    // reloads wait for every load in flight (64 x 4096 x 1024, f16 dst: 29.4 -> 25.4 us; the other types have the room and
    // lose 1 us to the arithmetic).  (The ring starts at a multiple of 128 bytes.)
    static constexpr bool ONE_ADDRESS = NS == 2;
    template <bool END = false>
    __device__ __forceinline__ void read_a1(int h, int i, int u, int slot) {
        const unsigned at = END && ONE_ADDRESS ? (ra[0][0] ^ (unsigned)(u << 6)) + slot * L::STAGE_BYTES : slot ? ra[1][u] : ra[0][u];
        a[h][i].c[u] = lds_read16(at + h * (64 * LKB) + i * (16 * LKB));
    }
    template <bool END = false>
    __device__ __forceinline__ void read_b1(int g, int j, int u, int slot) {
        const unsigned at = END && ONE_ADDRESS ? (rb[0][0] ^ (unsigned)(u << 6)) + slot * L::STAGE_BYTES : slot ? rb[1][u] : rb[0][u];
        b[g][j].c[u] = lds_read16(at + g * (L::WC / 2 * LKB) + j * (16 * LKB));
    }
    template <bool END>
    __device__ __forceinline__ void read_a(int h, int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 2; ++u) read_a1<END>(h, i, u, slot);
    }
    template <bool END>
    __device__ __forceinline__ void read_b(int g, int slot) {
#pragma unroll
        for (int j = 0; j < QC; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u) read_b1<END>(g, j, u, slot);
    }
    __device__ __forceinline__ void read_sa(int h, int slot) {
        if constexpr (NS > 0) {
            const int wm = G::wm(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
#pragma unroll
            for (int u = 0; u < NS; ++u) sa[h][u] = (int)lds_read4(rs + slot * Ld::SCALE_BYTES + (u * Ld::SG + wm * 2 + h) * 256);
        }
    }
    __device__ __forceinline__ void read_sb(int at, int slot) {
        if constexpr (NS > 0) {
            const int wn = G::wn(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
            static_assert(L::WC == 64 || NS == 0, "a group of 64 columns a wavefront");
#pragma unroll
            for (int u = 0; u < NS; ++u) sb[at][u] = (int)lds_read4(rs + slot * Ld::SCALE_BYTES + (u * Ld::SG + 4 + wn) * 256);
        }
    }
    // (chunks are whole but where K is any number of 16-bit elements)
    __device__ __forceinline__ void zero1(v4i &c, int u) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = inside[u] - 4 * e;
            c[e] = n >= 4 ? c[e] : (Ld::AKM && n == 2) ? c[e] & 0xffff : 0;
        }
    }
    __device__ __forceinline__ void zero(line_pair_t &f) const {
#pragma unroll
        for (int u = 0; u < 2; ++u) zero1(f.c[u], u);
    }
    // half t (4 of 8 k) of tile j's fragment for half u of the step, its lines across K
    __device__ __forceinline__ void read_bk1(int u, int j, int t, int slot) {
        const v2i_t x = lds_read_tr16(slot0 + slot * L::STAGE_BYTES + L::B_OFF + (kb ^ (unsigned)(j << 5)) + (u * 32 + t * 4) * Ld::BRB);
        b[j / QC][j % QC].c[u][2 * t] = x[0];
        b[j / QC][j % QC].c[u][2 * t + 1] = x[1];
    }
    __device__ __forceinline__ void read_ak1(int u, int h, int i, int t, int slot) {
        const v2i_t x = lds_read_tr16(slot0 + slot * L::STAGE_BYTES + (ka ^ (unsigned)((h * 4 + i) << 5)) + (u * 32 + t * 4) * Ld::ARB);
        a[h][i].c[u][2 * t] = x[0];
        a[h][i].c[u][2 * t + 1] = x[1];
    }
    __device__ __forceinline__ void read_bk(int u, int slot) {
#pragma unroll
        for (int j = 0; j < 2 * QC; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) read_bk1(u, j, t, slot);
    }
    __device__ __forceinline__ void read_ak(int u, int h, int slot) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t) read_ak1(u, h, i, t, slot);
    }
    __device__ __forceinline__ void ready_bk(int u, bool partial) {
        if (!partial) return;
#pragma unroll
        for (int j = 0; j < 2 * QC; ++j) zero1(b[j / QC][j % QC].c[u], u);
    }
    __device__ __forceinline__ void ready_ak(int u, int h, bool partial) {
        if (!partial) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) zero1(a[h][i].c[u], u);
    }
    // what fragments need between their read and their first product
    __device__ __forceinline__ void ready_a(int h, bool partial) {
#pragma unroll
        for (int i = 0; i < 4; ++i) Mma::prepare_a(a[h][i]);
        if (partial) {
#pragma unroll
            for (int i = 0; i < 4; ++i) zero(a[h][i]);
        }
    }
    __device__ __forceinline__ void ready_b(int g, bool partial) {
#pragma unroll
        for (int j = 0; j < QC; ++j) Mma::prepare_b(b[g][j]);
        if (partial) {
#pragma unroll
            for (int j = 0; j < QC; ++j) zero(b[g][j]);
        }
    }
};

// f(0), f(1), ... with the index as a constant expression
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<N, I + 1>(f);
    }
}

// Eight wavefronts, two per SIMD, in two groups of four that alternate: while one group multiplies a quadrant, the
// other reads the fragments of its next one and issues loads, and a barrier ends every such phase.  Two wavefronts of
// a SIMD that multiply at the same time, with reads and loads spread between the MFMAs and a barrier a phase or two a
// step, measured the same (bf16 8192^3 0.7205 / 0.7208 ms, int8 0.371 / 0.371) on 250 registers instead of 212; what
// the registers leave is what the fused epilogues and block scales live on.
//
// Phases of step s (its slot s % 2): what is read, what is loaded into the part that the phase before released
//   0  B half 0, A half 0, scales   A half 1 of step s + 1
//   1  B half 1                     B half 0 and the scales of step s + 2
//   2  A half 1                     A half 0 of step s + 2
//   3                               B half 1 of step s + 2
// A wavefront has its reads back before the barrier that ends the phase's reading part, so a released part is free
// for both groups.  A part is complete once every wavefront's own loads of it have landed before a barrier ahead of the
// phase that reads it: the counts below are what a wavefront has issued after them.
template <class Mma, class Acc, class Fill>
__device__ __forceinline__ void main_loop_lines8(Acc &acc, char *smem, const char *a_tile, const char *b_tile, long lda,
        long ldb, long rows_a_left, long rows_b_left, long kbytes, const line_scales_t &sc, Fill &&fill) {
    using Ld = line_loader_t<Mma>;
    using Fr = line_frags_t<Mma>;
    using G = typename Mma::G;
    static_assert(G::NW == 8, "two groups of four wavefronts");
    constexpr int DA = Ld::L::DPA, DB = Ld::L::DPB, EX = Ld::EX, QC = Fr::QC, NU = Mma::NU;
    Ld ld;
    ld.init(smem, a_tile, b_tile, lda, ldb, rows_a_left, rows_b_left, kbytes, sc);
    Fr f;
    f.init(ld, kbytes);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool late = wave >= 4;

    auto quadrant = [&](auto H, auto Gc) __attribute__((always_inline)) {
        constexpr int h = decltype(H)::value, g = decltype(Gc)::value;
        __builtin_amdgcn_s_setprio(1);
        static_for<NU>([&](auto U) __attribute__((always_inline)) {
            static_for<4>([&](auto I) __attribute__((always_inline)) {
                static_for<QC>([&](auto J) __attribute__((always_inline)) {
                    constexpr int u = decltype(U)::value, i = decltype(I)::value, j = decltype(J)::value;
                    Mma::template mma<g * QC + j, i>(acc[h * 4 + i][g * QC + j], f.b[g][j], f.a[h][i], U,
                            f.sb[0][Fr::NS ? u : 0], f.sa[h][Fr::NS ? u : 0]);
                });
            });
        });
        __builtin_amdgcn_s_setprio(0);
    };
    constexpr std::integral_constant<int, 0> c0 {};
    constexpr std::integral_constant<int, 1> c1 {};
    // Operands with their lines across K (B, or both): a quadrant is a half of the rows and a half of the 64 k, and what a
    // phase reads follows: B half 0 and A half 0 | B half 1 | A half 1 | -  becomes, with k halves,
    //   B only   B k 0 and A rows 0 | B k 1 | A rows 1 | -
    //   both     B k 0 and A k 0, rows 0 | A k 0, rows 1 | B k 1 and A k 1, rows 0 | A k 1, rows 1
    // The schedule of the loads, and with it the counts, are the same.
    constexpr bool AKM = Ld::AKM, BKM = Ld::BKM;
    static_assert(BKM || !AKM, "src across K comes with weights across K");
    auto quadrant_k = [&](auto H, auto U) __attribute__((always_inline)) {
        constexpr int h = decltype(H)::value, u = decltype(U)::value;
        __builtin_amdgcn_s_setprio(1);
        static_for<4>([&](auto I) __attribute__((always_inline)) {
            static_for<2 * QC>([&](auto J) __attribute__((always_inline)) {
                constexpr int i = decltype(I)::value, j = decltype(J)::value;
                Mma::template mma<j, i>(acc[h * 4 + i][j], f.b[j / QC][j % QC], f.a[h][i], std::integral_constant<int, u>(), 0, 0);
            });
        });
        __builtin_amdgcn_s_setprio(0);
    };
    auto products = [&](auto First, auto Second) __attribute__((always_inline)) {
        if constexpr (AKM) quadrant_k(Second, First);
        else if constexpr (BKM) quadrant_k(First, Second);
        else quadrant(First, Second);
    };

    ld.template load_scales<true>(0, 0);
    ld.template load_b<true>(0, 0, 0);
    ld.template load_a<true>(0, 0, 0);
    ld.template load_b<true>(1, 0, 0);
    ld.template load_a<true>(1, 0, 0);
    ld.template load_b<true>(0, 1, 1);
    ld.template load_scales<true>(1, 1);
    ld.template load_a<true>(0, 1, 1);
    ld.template load_b<true>(1, 1, 1);
    fill();
    constexpr int STEP = 2 * DA + 2 * DB + EX; // loads of a step
    wait_vmcnt<STEP + DB>();                   // after A 0 of step 0: B 1, A 1, then step 1 without its A 1
    phase_barrier();
    if (late) phase_barrier();
    auto step = [&](auto End, int s, int slot) __attribute__((always_inline)) {
        constexpr bool END = decltype(End)::value;
        const bool partial = END && ld.tail_mask != 0 && s == ld.nst - 1;
        f.read_sb(0, slot);
        if constexpr (BKM) f.read_bk(0, slot);
        else f.template read_b<END>(0, slot);
        f.read_sa(0, slot);
        f.read_sa(1, slot);
        if constexpr (AKM) f.read_ak(0, 0, slot);
        else f.template read_a<END>(0, slot);
        ld.template load_a<END>(1, s + 1, slot ^ 1);
        wait_vmcnt<STEP + DA>(); // after B 1 of s: A 1, then all of s + 1
        wait_lds_reads();
        if constexpr (BKM) f.ready_bk(0, partial);
        else f.ready_b(0, partial);
        if constexpr (AKM) f.ready_ak(0, 0, partial);
        else f.ready_a(0, partial);
        phase_barrier();
        products(c0, c0);
        phase_barrier();
        if constexpr (AKM) f.read_ak(0, 1, slot);
        else if constexpr (BKM) f.read_bk(1, slot);
        else f.template read_b<END>(1, slot);
        ld.template load_b<END>(0, s + 2, slot);
        ld.template load_scales<END>(s + 2, slot);
        wait_vmcnt<STEP + DB + EX>(); // after A 1 of s: all of s + 1, B 0 and scales of s + 2
        wait_lds_reads();
        if constexpr (AKM) f.ready_ak(0, 1, partial);
        else if constexpr (BKM) f.ready_bk(1, partial);
        else f.ready_b(1, partial);
        phase_barrier();
        products(c0, c1);
        phase_barrier();
        if constexpr (AKM) {
            f.read_bk(1, slot);
            f.read_ak(1, 0, slot);
        } else {
            f.template read_a<END>(1, slot);
        }
        ld.template load_a<END>(0, s + 2, slot);
        wait_lds_reads();
        if constexpr (AKM) {
            f.ready_bk(1, partial);
            f.ready_ak(1, 0, partial);
        } else {
            f.ready_a(1, partial);
        }
        phase_barrier();
        if constexpr (BKM) products(c1, c0);
        else products(c1, c1);
        phase_barrier();
        if constexpr (AKM) f.read_ak(1, 1, slot);
        ld.template load_b<END>(1, s + 2, slot);
        wait_vmcnt<STEP + DB>(); // after A 0 of s + 1: B 1 and A 1 of s + 1, s + 2 without its A 1
        if constexpr (AKM) {
            wait_lds_reads();
            f.ready_ak(1, 1, partial);
        }
        phase_barrier();
        if constexpr (BKM) products(c1, c1); // (every sum takes its k in the order that copied operands give)
        else products(c1, c0);
        phase_barrier();
    };
    int s = 0;
    const int steady = ld.steady();
#pragma nounroll
    for (; s + 1 < steady; s += 2) {
        step(std::false_type {}, s, 0);
        step(std::false_type {}, s + 1, 1);
    }
#pragma nounroll
    for (; s < ld.nst; ++s) step(std::true_type {}, s, s & 1);
    if (!late) phase_barrier();
    // every load has landed (the clamped ones included) before the ring's memory is used for something else
    wait_vmcnt<0>();
    phase_barrier();
}

// Four wavefronts, one per SIMD, for the 256 x 128 tile.  Nobody covers for a wavefront that waits, so nothing a
// quadrant needs is requested in it: the fragments of the next half step are read between the MFMAs of this one, and
// the loads with them.  One wavefront with 128 accumulators keeps a matrix core as busy as two of the eight-wavefront
// tile (bf16 2048 x 4096 x 14336, 256 tiles: 168 us; the same tile on eight wavefronts of 128 x 32, which read 1.7
// times as much from LDS, 212 us; the 64-byte steps that this loop took the place of 247).
//
// A step s is two halves:
//          products              reads                     loads
//   X(s)   (A 0, B 0) (A 0, B 1)   B 1, A 1 of step s        B 0, A 0 of step s + 2
//   Y(s)   (A 1, B 0) (A 1, B 1)   A 0, B 0 of step s + 1    scales, B 1, A 1 of step s + 2
// with one barrier before each: every read of the half before is back, so what it read may be loaded again, and what
// this one reads landed (loads of four parts have been issued after it).
//
// The MFMAs are inline assembly with the accumulator tied to one operand: left to itself the compiler accumulates out
// of place in the two-fold unrolled loop and moves 192 accumulator registers a step.  The accumulators are accumulation
// registers, of which nothing else wants any: among the plain ones the allocator parked a few elsewhere between steps, and
// what it read right behind an MFMA that it does not know as one was not written yet.  A VALU result needs two wait
// states before an MFMA reads it, which the compiler cannot place either (s_nop below).
template <class Mma, class Acc, class Fill>
__device__ __forceinline__ void main_loop_lines4(Acc &acc, char *smem, const char *a_tile, const char *b_tile, long lda,
        long ldb, long rows_a_left, long rows_b_left, long kbytes, const line_scales_t &sc, Fill &&fill) {
    using Ld = line_loader_t<Mma>;
    using Fr = line_frags_t<Mma>;
    constexpr bool BKM = Ld::BKM; // weights across K: a column half is a half of the 64 k instead
    static_assert(Mma::G::NW == 4 && !Ld::AKM, "four wavefronts");
    constexpr int DA = Ld::L::DPA, DB = Ld::L::DPB, EX = Ld::EX, QC = Fr::QC, NU = Mma::NU, NS = Fr::NS;
    Ld ld;
    ld.init(smem, a_tile, b_tile, lda, ldb, rows_a_left, rows_b_left, kbytes, sc);
    Fr f;
    f.init(ld, kbytes);

    ld.template load_a<true>(0, 0, 0);
    ld.template load_b<true>(0, 0, 0);
    ld.template load_scales<true>(0, 0);
    ld.template load_b<true>(1, 0, 0);
    ld.template load_a<true>(1, 0, 0);
    ld.template load_b<true>(0, 1, 1);
    ld.template load_a<true>(0, 1, 1);
    ld.template load_scales<true>(1, 1);
    ld.template load_b<true>(1, 1, 1);
    ld.template load_a<true>(1, 1, 1);
    fill();
    wait_vmcnt<3 * (DA + DB) + EX>();
    phase_barrier();
    f.read_sb(0, 0);
    f.read_sa(0, 0);
    f.template read_a<false>(0, 0);
    if constexpr (BKM) f.read_bk(0, 0);
    else f.template read_b<false>(0, 0);

    // two wait states behind everything that ready_a / ready_b compute (the scheduler would sink it to its use)
    auto settle = []() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 1");
        __builtin_amdgcn_sched_barrier(0);
    };
    // First: X, otherwise Y; slot of step s
    auto half = [&](auto End, auto First, int s, int slot) __attribute__((always_inline)) {
        constexpr bool END = decltype(End)::value, first = decltype(First)::value;
        constexpr int h = first ? 0 : 1, read_half = 1 - h, load_half = h;
        const int rslot = first ? slot : slot ^ 1;
        const bool partial = END && ld.tail_mask != 0 && s == ld.nst - 1;
        wait_vmcnt<2 * (DA + DB) + (first ? EX : 0)>(); // (the scales go in front of Y's loads)
        wait_lds_reads();
        phase_barrier();
        if (first) {
            f.read_sa(1, slot);
        } else {
            f.read_sa(0, slot ^ 1);
            f.read_sb(slot ^ 1, slot ^ 1);
            ld.template load_scales<END>(s + 2, slot);
        }
        f.ready_a(h, partial);
        auto ready_cols = [&](int g) __attribute__((always_inline)) {
            if constexpr (BKM) f.ready_bk(g, partial);
            else f.ready_b(g, partial);
        };
        if (first) ready_cols(0);
        settle();
        constexpr int NB = BKM ? 4 * QC : 2 * QC, NR = NB + 8, NM = BKM ? 8 * QC : 4 * QC * NU, ND = DA + DB;
        constexpr int PER = NM >= 16 ? 1 : 2; // reads ahead of an MFMA
        int n = 0, read = 0, loaded = 0;
        static_for<2>([&](auto Qd) __attribute__((always_inline)) {
            constexpr int qd = decltype(Qd)::value;
            if (first && qd == 1) {
                ready_cols(1);
                settle();
            }
            static_for<BKM ? 1 : NU>([&](auto U) __attribute__((always_inline)) {
            static_for<4>([&](auto I) __attribute__((always_inline)) {
            static_for<BKM ? 2 * QC : QC>([&](auto J) __attribute__((always_inline)) {
                constexpr int u = BKM ? qd : decltype(U)::value, i = decltype(I)::value;
                constexpr int j = BKM ? decltype(J)::value : qd * QC + decltype(J)::value; // column tile
#pragma unroll
                for (int p = 0; p < PER; ++p) {
                    // X: the columns first, its second quadrant wants them; Y: they replace its first quadrant's
                    const bool cols = first ? read < NB : read >= 8;
                    if (read < NR && (first || !cols || qd == 1)) {
                        const int e = first ? (cols ? read : read - NB) : (cols ? read - 8 : read);
                        if (!cols) f.read_a1(read_half, e / 2, e % 2, rslot);
                        else if (BKM) f.read_bk1(read_half, e / 2, e % 2, rslot);
                        else f.read_b1(read_half, e / 2, e % 2, rslot);
                        ++read;
                    }
                }
                if (loaded < ND && n == (2 * loaded + 1) * NM / ND) {
                    if (loaded < DB) ld.template load_b1<END>(load_half, loaded, s + 2, slot);
                    else ld.template load_a1<END>(load_half, loaded - DB, s + 2, slot);
                    ++loaded;
                }
                Mma::template mma_tied<j, i>(acc[h * 4 + i][j], f.b[j / QC][j % QC], f.a[h][i], u, f.sb[slot][NS ? u : 0],
                        f.sa[h][NS ? u : 0]);
                __builtin_amdgcn_sched_barrier(0); // keeps the reads and loads spread between the MFMAs
                ++n;
            });
            });
            });
        });
    };
    auto step = [&](auto End, int s, int slot) __attribute__((always_inline)) {
        half(End, std::true_type {}, s, slot);
        half(End, std::false_type {}, s, slot);
    };
    int s = 0;
    const int steady = ld.steady();
#pragma nounroll
    for (; s + 1 < steady; s += 2) {
        step(std::false_type {}, s, 0);
        step(std::false_type {}, s + 1, 1);
    }
#pragma nounroll
    for (; s < ld.nst; s += 2) {
        step(std::true_type {}, s, 0);
        if (s + 1 < ld.nst) step(std::true_type {}, s + 1, 1);
    }
    // every load has landed and every read is back before the ring's memory is used for something else; the wait
    // states between the last MFMA and the first read of its result
    wait_vmcnt<0>();
    wait_lds_reads();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    phase_barrier();
}

// fill(): what the kernel prepares for its epilogue; its loads wait behind the first steps' and not in front of them
// (1.5 us a tile)
template <class Mma, class Acc, class Fill>
__device__ __forceinline__ void main_loop_lines(Acc &acc, char *smem, const char *a_tile, const char *b_tile, long lda,
        long ldb, long rows_a_left, long rows_b_left, long kbytes, const line_scales_t &sc, Fill &&fill) {
    if constexpr (Mma::G::NW == 8)
        main_loop_lines8<Mma>(acc, smem, a_tile, b_tile, lda, ldb, rows_a_left, rows_b_left, kbytes, sc, fill);
    else
        main_loop_lines4<Mma>(acc, smem, a_tile, b_tile, lda, ldb, rows_a_left, rows_b_left, kbytes, sc, fill);
}

// operand policies of these loops
template <class Mma, class = void>
struct reads_lines : std::false_type {};
template <class Mma>
struct reads_lines<Mma, std::enable_if_t<(Mma::NU > 0)>> : std::true_type {};

// Which of the two tiles a problem of `batch` x M x N takes: rounds of 256 workgroups, one a CU.  A round of 256 x 128 tiles
// is the cheaper one, so no more of them than of large ones are taken always.  Three against two take as long or less
// only where K is long, 9 / 16 of the time for a round (bf16 / int8 / fp8, K = 4096: 39 / 23.4 / 22.7 us against 69 / 40 / 39),
// and the epilogue is a chain: 4096 x 5120, narrow against wide, bf16 with K = 256 / 1024 / 4096 32.5 / 29.3, 56.9 / 56.9, 149 / 164
// us, fp8 with K = 1024 / 4096 42.7 / 40.9, 89.8 / 94.2, and through the general epilogue 69.8 / 59.1, 116 / 111.  Beyond two
// rounds of large tiles the chip is power-limited and the small tile's 1.5 loads per MFMA cost 10 %.
// (N up to 128, half of a large tile at most, has stayed on them since the tiles were chosen by count alone.  The narrow one
// measures 0.66 to 0.89 of their time there, fp8: 4096 x 128 x 1024 13.4 / 17.5 us, 70000 x 100 x 2048 96.5 / 108.)
inline bool line_tiles_narrow(long batch, long M, long N, long kbytes, bool chain) {
    if (N <= 128) return false;
    const long tm = (M + BM - 1) / BM, wide = batch * tm * ((N + 255) / 256), narrow = batch * tm * ((N + 127) / 128);
    const long rounds_wide = (wide + 255) / 256, rounds_narrow = (narrow + 255) / 256;
    return wide <= 512 && (rounds_narrow <= rounds_wide || (chain && kbytes >= 4096 && 9 * rounds_narrow < 16 * rounds_wide));
}

} // namespace gemm
} // namespace mi355
