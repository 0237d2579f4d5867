// The tiles of the GEMM families: geometry, tile order, and the K loop of the f32 type.
//
// Shape of the computation: one workgroup = one 256 x 256 dst tile of eight wavefronts (128 x 64 each, 128 accumulator
// registers, two wavefronts per SIMD), or a 256 x 128 tile of four.  Both operands are consumed K-contiguous ("A" rows
// are src rows, "B^T" rows are weight columns):
//
//   HBM/L2 --global_load_lds_dwordx4--> LDS ring (the loads bypass the register file)
//   LDS --ds_read_b128--> MFMA operands --v_mfma--> accumulators
//   accumulators --fused epilogue--> dst stores (the MFMA operands are exchanged, so a lane holds four consecutive n of
//       a row)
//
// The loads are inline assembly so that the outstanding-load counter is managed by hand.  The loops of all types but
// f32 are in line_loops.hpp: 128 bytes of K a step.  f32 takes eight times the matrix cycles per byte, is bound by its
// instruction (91 % of its peak) and keeps stages of 64 bytes, which its 32 x 32 fragments are laid out for.
#pragma once
#include "kernels.hpp"
#include "tile_epilogue.hpp"

namespace mi355 {

namespace gemm {

constexpr int BM = 256;               // rows of a workgroup's dst tile
constexpr int BKB = 64;               // bytes of K per row per stage
constexpr int B_OFF = BM * BKB;       // B^T tile offset inside a stage

// Tile geometry: a workgroup of NW wavefronts computes a 256 x BN dst tile, two wavefronts along m (128 rows each) and
// NW/2 along n.  The stage members describe the 64-byte stages of the f32 loop.
template <int NW_, int BN_>
struct geo_t {
    static constexpr int NW = NW_, NT = 64 * NW_, BN = BN_;
    static constexpr int WN = NW_ / 2;        // wavefronts along n
    static constexpr int WCOLS = BN_ / WN;    // columns of a wavefront's part
    static constexpr int DPA = (BM / 16) / NW_;  // A DMAs per stage and wavefront
    static constexpr int DPB = (BN_ / 16) / NW_; // B^T DMAs per stage and wavefront
    static constexpr int DPS = DPA + DPB;
    static constexpr int STAGE_BYTES = (BM + BN_) * BKB;
    static constexpr int NSTAGE = 4; // ring depth
    __device__ static __forceinline__ int wm(int wave) { return wave / WN; }
    __device__ static __forceinline__ int wn(int wave) { return wave % WN; }
};

// Chunk swizzle.  Measured on MI355X with a read-only micro-benchmark over all
// XOR-of-row-bits functions: this one is free of bank conflicts for both
// fragment read patterns of 64-byte rows (16 rows x 4 chunks across the 64
// lanes; 32 rows x 2 chunks in two reads, what the f32 tiles' 32x32 shape reads),
// where e.g. ((row >> 1) & 3) ^ ((row >> 3) & 1) costs the 16-row one a factor of two.
__device__ __forceinline__ int swz_f(int row) {
    return ((row >> 2) & 1) | ((((row >> 2) ^ (row >> 3)) & 1) << 1);
}
__device__ __forceinline__ int swz(int row, int chunk) {
    return row * BKB + ((chunk ^ swz_f(row)) << 4);
}

struct tile_pos_t {
    long m0, n0;
};

// XCD-aware tile order.  Consecutive workgroup ids land on different XCDs
// (8 of them, each with a private L2); give every XCD one contiguous run of
// tiles, walked in bands of GM tile rows so that concurrently resident tiles
// share A rows and B columns in that L2.
// (A persistent form, one workgroup per CU walking ids blockIdx.x + k * gridDim.x,
// measured the same as one workgroup per tile: the turnover between tiles is
// ~6 us of 130.)
template <class G>
__device__ __forceinline__ tile_pos_t tile_position(int id, int tiles_m, int tiles_n) {
    const int nwg = tiles_m * tiles_n;
    const int per = nwg / 8;
    const int tile = (nwg % 8 == 0) ? (id % 8) * per + id / 8 : id;
    constexpr int GM = 8; // measured: 4 and 8 alike, 16 is 2 % and 32 is 7 % slower on the int8 headline shape
    const int band = tile / (GM * tiles_n);
    const int band_rows = min(GM, tiles_m - band * GM);
    const int in_band = tile - band * GM * tiles_n;
    tile_pos_t p;
    p.m0 = (long)(band * GM + in_band % band_rows) * BM;
    p.n0 = (long)(in_band / band_rows) * G::BN;
    return p;
}

// Per-thread DMA plan: wave w owns DPA blocks of 16 tile rows of A and DPB of
// B^T, one DMA each per stage.
template <int DPA, int DPB>
struct dma_plan_t {
    unsigned voff_a[DPA], voff_b[DPB]; // byte offsets from the scalar tile base
    unsigned lds_a[DPA], lds_b[DPB];   // LDS byte offsets inside a stage
};

template <int DPA, int DPB>
__device__ __forceinline__ dma_plan_t<DPA, DPB> make_dma_plan(int wave, int lane, long rows_a_left,
        long rows_b_left, long lda, long ldb) {
    dma_plan_t<DPA, DPB> p;
#pragma unroll
    for (int i = 0; i < DPA; ++i) {
        const int row = (wave * DPA + i) * 16 + (lane >> 2);
        const int chunk = (lane & 3) ^ swz_f(row);
        long ra = row;
        if (ra > rows_a_left - 1) ra = rows_a_left - 1;
        p.voff_a[i] = (unsigned)(ra * lda + chunk * 16);
        p.lds_a[i] = (unsigned)((wave * DPA + i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < DPB; ++i) {
        const int row = (wave * DPB + i) * 16 + (lane >> 2);
        const int chunk = (lane & 3) ^ swz_f(row);
        long rb = row;
        if (rb > rows_b_left - 1) rb = rows_b_left - 1;
        p.voff_b[i] = (unsigned)(rb * ldb + chunk * 16);
        p.lds_b[i] = (unsigned)(B_OFF + (wave * DPB + i) * 1024);
    }
    return p;
}

// Main loop for eight wavefronts, two per SIMD, in two groups of four that run
// half a K step apart.  Both groups meet at one workgroup barrier per step; in
// the interval after barrier g
//   group 0:  reads stage g from LDS, then its MFMAs of stage g
//   group 1:  its MFMAs of stage g-1 (fragments read in the previous interval),
//             then reads stage g
// so on every SIMD one wavefront has MFMAs to issue while the other one waits
// for LDS, with every wavefront's instruction stream in plain program order:
// nothing depends on how the compiler interleaves reads with MFMAs.  Both
// groups read stage g in the same interval, so one barrier per step covers
// both conditions: every wavefront waits for its own DMAs of stage g before
// barrier g (then all of stage g is in LDS), and has its reads of stage g-1
// back before it (then that slot may be overwritten by the DMAs of stage
// g+NG-1, which are issued after the barrier).  Group 1 runs one more
// iteration for its last MFMAs.
template <int NSTAGE, class Mma, class Acc>
__device__ __forceinline__ void main_loop_two_groups(Acc &acc, char *smem, const char *a_tile_,
        const char *b_tile_, long lda, long ldb, long rows_a_left, long rows_b_left, int ngroups_) {
    using G = typename Mma::G;
    const char *a_tile = scalar_ptr(a_tile_), *b_tile = scalar_ptr(b_tile_);
    // (a uniform value merged from two loads at the join of divergent code ahead of
    // the loop counts as divergent, and the stage offsets derive from it)
    const int ngroups = scalar_int(ngroups_);
    static_assert(G::NW == 8, "two groups of four wavefronts");
    constexpr int NG = NSTAGE;
    constexpr int STAGE_BYTES = G::STAGE_BYTES;
    constexpr int DPA = G::DPA, DPB = G::DPB, DPS = G::DPS;
    constexpr int GROUP_DMAS = DPS;
    static_assert(NG >= 3 && NG <= 5, "ring depth");
    static_assert((NG - 2) * GROUP_DMAS < 64, "vmcnt range");
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const typename Mma::addr_t AD = Mma::lane_addr(G::wm(wave), G::wn(wave), lane);
    const bool late = wave >= 4; // group 1
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) char *)smem;
    const dma_plan_t<DPA, DPB> plan = make_dma_plan<DPA, DPB>(wave, lane, rows_a_left, rows_b_left, lda, ldb);

    auto issue_part = [&](int g, int slot, int i) __attribute__((always_inline)) {
        const long koff = (long)g * BKB;
        const unsigned lds_stage = lds0 + slot * STAGE_BYTES;
        if (i < DPA) dma16(a_tile + koff, plan.voff_a[i], lds_stage + plan.lds_a[i]);
        else dma16(b_tile + koff, plan.voff_b[i - DPA], lds_stage + plan.lds_b[i - DPA]);
    };
    // the MFMAs of one stage with the DMAs of stage gd spread between the rows:
    // a DMA instruction can wait tens of cycles for the address unit, which
    // passes unnoticed behind a row of MFMAs
    // Past the last stage the DMAs are issued all the same, clamped to the last
    // stage and into a slot nobody reads again: the MFMA sequence stays one
    // basic block (conditional blocks between the rows make the register
    // allocator spill accumulators), and every stage is followed by the same
    // number of loads, so one outstanding-load count fits every iteration.
    auto mma_stage = [&](const typename Mma::frag_t &f, int gd, int dslot) __attribute__((always_inline)) {
        const int gdc = gd < ngroups ? gd : ngroups - 1;
#pragma unroll
        for (int i = 0; i < Mma::ROWS; ++i) {
            Mma::mma_row(acc, f, i);
#pragma unroll
            for (int d = 0; d < DPS; ++d)
                if (d * Mma::ROWS / DPS == i) issue_part(gdc, dslot, d);
            __builtin_amdgcn_sched_barrier(0); // or the DMAs all move to the front
        }
    };

#pragma unroll
    for (int s = 0; s < NG - 1; ++s) {
        const int sc = s < ngroups ? s : ngroups - 1;
#pragma unroll
        for (int i = 0; i < DPS; ++i) issue_part(sc, s, i);
    }

    int slot = 0;
    // Group 1 carries the fragments from one iteration to the next; they start
    // as zeros (Mma::zero_frag), so that its first iteration, which has no stage to multiply yet, adds zero
    // products instead of branching around the MFMAs (one MFMA sequence on every
    // path keeps the accumulators where they are).
    typename Mma::frag_t f = Mma::zero_frag();
    const int niter = ngroups + (late ? 1 : 0);
    auto read_stage = [&]() __attribute__((always_inline)) {
        const unsigned S = lds0 + slot * STAGE_BYTES;
        Mma::load_a(f, 0, S, AD);
        Mma::load_b(f, S, AD);
#pragma unroll
        for (int i = 1; i < Mma::ROWS; ++i) Mma::load_a(f, i, S, AD);
    };
#pragma nounroll
    for (int g = 0; g < niter; ++g) {
        // own DMAs of stage g landed; those of NG-2 later stages may stay in flight
        wait_vmcnt<(NG - 2) * GROUP_DMAS>();
        if (late) wait_lds_reads();
        phase_barrier();
        int nslot = slot + NG - 1; // the slot stage g-1 used: free after this barrier
        if (nslot >= NG) nslot -= NG;
        if (!late) read_stage();
        __builtin_amdgcn_sched_barrier(0);
        // Group 1 gets the matrix core first: its MFMAs were ready at the barrier,
        // and its reads for the next interval come after them.  At equal priority
        // group 0, which starts ~125 ns later, is served first all the same and
        // group 1's reads end up after all MFMAs of the step, with the matrix core
        // idle (time stamps: 545 ns for group 1's block against 285 ns for group 0's;
        // with the priority 300 against 480, and 1.5-2 % less time per launch).
        if (late) __builtin_amdgcn_s_setprio(3);
        mma_stage(f, g + NG - 1, nslot); // group 0: stage g; group 1: stage g-1
        if (late) __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        if (late && g < ngroups) read_stage();
        if (++slot == NG) slot = 0;
    }
    if (!late) phase_barrier(); // the barrier of group 1's last iteration
    // every DMA has landed (the clamped ones included) before the ring's memory
    // is used for something else
    wait_vmcnt<0>();
    phase_barrier();
}

} // namespace gemm
} // namespace mi355
