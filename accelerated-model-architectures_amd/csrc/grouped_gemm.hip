// Grouped (per-expert, ragged) GEMMs of the MoE layer on CDNA4 MFMA.
//
// One workgroup = 256 threads = 4 wave64 (2 x 2), output tile 256 x 256, K step 64.  Each wave owns 128 x 128 =
// 4 x 4 v_mfma_f32_32x32x16 tiles (256 fp32 accumulators per lane, one wave per SIMD).
//
// Operand tiles go from HBM straight into LDS with global_load_lds_dwordx4 (no VGPR staging, no ds_write): a wave
// instruction moves 64 x 16 bytes to 1 KB of consecutive LDS, and the swizzle is applied on the GLOBAL side (which
// lane fetches which 16-byte chunk).  Every such instruction covers whole 128-byte lines (8 per instruction): the
// texture addresser works line by line, and half-line requests (a 32-wide K step) were measured at a third of the
// throughput.  Two LDS layouts, both 32 KB per 256 x 64 operand tile:
//   row-major source (K contiguous in memory):  LDS [256 rows][8 chunks], chunk c of row r at slot c ^ swz(r);
//       MFMA fragments are one ds_read_b128 per lane.
//   transposed source (K is the row index in memory: weights for dX, both operands for dW):
//       LDS [64 k][32 chunks] exactly as in memory, chunk c of k-row kr at slot c ^ ((kr & 3) << 1);
//       MFMA fragments are two ds_read_b64_tr_b16 per lane, which hand each lane 4 consecutive k of one column.
//
// Pipeline: two stages (128 KB of the 160 KB LDS).  The persistent forward / dX kernel walks a K step by quadrants of the
// tile (below, at "K loop by quadrants").  The others have one barrier per K step, which is four k16 sub-steps of 16 MFMAs;
// the fragments of sub-step kk + 1 are read while sub-step kk multiplies.  The barrier sits between sub-steps 2 and 3:
// by then a wave holds the last fragments of the step in registers, so behind the barrier the other stage (step s + 1,
// waited for with vmcnt(0) just before) is readable and this stage is free.  The loads of step s + 2 are issued one per
// MFMA slot during sub-steps 0 and 1 of step s + 1, which leaves them a step and a half to land.  A wave issues in
// order, so everything that is not an MFMA is pinned between MFMAs (sched_barrier) instead of in front of them.
//
// MFMA operand roles: the "P" tile supplies the rows of the 32x32 result (register dimension: a lane holds 4
// consecutive P indices per accumulator quad) and the "Q" tile supplies its columns (lane % 32).  P is always the
// dimension that is contiguous in the OUTPUT, so a lane stores 8 contiguous bytes per quad and owns one output row:
// gather/scatter indices, row scales and the SwiGLU (gate, up) pairs are all lane-local.
//
//   forward / dX :  Q = activation rows (tokens),     P = weight rows (output features)
//   dW           :  Q = dY columns (out features),    P = X columns (in features), K = tokens
//
// Tiles never straddle experts: the schedule is expert-major, derived on the device from the inclusive expert
// offsets in each workgroup's prologue (no host read of the counts).  With a workspace, the tiles of a last, partial
// round of a launch are computed as K slices by a second launch and summed by grouped_gemm_fixup_kernel.
//
// Epilogues (plain store with optional row scale and scatter, SwiGLU forward, SwiGLU backward) stage every 32-row block
// of a wave's corner in wave-private LDS and write whole rows: in the accumulator layout a store instruction would
// touch 32 rows with 16 bytes each.
#include <atomic>

#include "fp32.hpp"
#include "grouped_gemm_tile.hpp"
#include "k_schedule.hpp"

namespace xma_rocm {

constexpr int BK = 64, NSTAGE = 2;
// The 16 LDS-DMA pieces of a K step are issued one per MFMA slot: DMA_N0 in the sub-step right behind the barrier that
// frees their stage, DMA_N1 and DMA_N2 in the two sub-steps after it.
// (8, 8, 0) measured best; (6, 6, 4), (12, 4, 0) the same within noise, all 16 in the first sub-step slower.
constexpr int DMA_N0 = 8, DMA_N1 = 8, DMA_N2 = 0;
static_assert(DMA_N0 + DMA_N1 + DMA_N2 == 16 && DMA_N0 <= 16 && DMA_N1 <= 8 && DMA_N2 <= 8, "piece schedule");
constexpr int OP_CHUNKS = 256 * 8;                          // 16-byte chunks per operand tile (32 KB)
constexpr int STAGE_CHUNKS = 2 * OP_CHUNKS;                 // Q tile then P tile
constexpr int GEMM_SMEM_BYTES = NSTAGE * STAGE_CHUNKS * 16; // 128 KB

// 1 KB of zeros: the source of every chunk that lies beyond the K extent of an operand
__device__ __attribute__((aligned(16))) uint32_t g_zero_page[256];

__device__ __forceinline__ void lds_dma16(const uint16_t *src, u32x4 *lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)lds_wave_base, 16, 0, 0);
}

// ---- LDS layouts (byte offsets inside one 32 KB operand tile)
//
// The LDS serves 16 lanes of a ds_read_b128 (32 lanes of a 64-bit read) at a time from 64 banks of 4 bytes, so the 16-byte
// pieces those lanes ask for must fall on 16 different positions modulo 256 bytes.  Both layouts below are arranged for
// that (measured with the fragment patterns alone, 4 waves per CU: 344 bytes/ns/CU against 281 for swizzles that only
// spread 8 consecutive lanes over 128 bytes).
//
// Row-major tile [256 rows][8 chunks of 16 B]: chunk c of row r sits at slot c ^ ((r >> 1) & 7); rows 2 m and 2 m + 1
// share the permutation and are 128 bytes apart.  An LDS-DMA instruction covers 8 rows (1 KB); wave w loads rows
// 64 w + 8 i + (lane >> 3), i = 0..7, and lane fills slot lane & 7, i.e. it fetches logical chunk
// (lane & 7) ^ (4 (i & 1) + (lane >> 4)): one of two per-lane constants, so a lane's global address of piece i is a fixed
// per-lane pointer plus the K offset of the step.
__device__ __forceinline__ int rowmajor_lane_chunk(int i, int lane) { return (lane & 7) ^ (((i & 1) << 2) + (lane >> 4)); }
// MFMA fragment of rows R0 + 32 i + (lane & 31), k16 sub-step kk: R0 and 32 i are multiples of 16, so the slot is
// ((2 kk + (lane >> 5)) ^ ((lane >> 1) & 7)): one per-lane byte offset per kk, and i is an immediate (4096 i).
__device__ __forceinline__ uint32_t rowmajor_frag_offset(int R0, int kk, int lane) {
    return (uint32_t)((R0 + (lane & 31)) * 128 + (((2 * kk + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4));
}
//
// Transposed tile [64 k-rows][32 chunks of 16 B], exactly as in memory: chunk c of k-row kr sits at slot
// c ^ ((kr & 3) << 2).  An LDS-DMA instruction covers 2 k-rows; wave w loads k-rows 16 w + 2 j + (lane >> 5), j = 0..7,
// and lane fills slot lane & 31, i.e. it fetches logical chunk (lane & 31) ^ (((2 j + (lane >> 5)) & 3) << 2).
__device__ __forceinline__ int transposed_lane_chunk(int j, int lane) {
    return (lane & 31) ^ (((2 * j + (lane >> 5)) & 3) << 2);
}
// MFMA fragment through ds_read_b64_tr_b16, which works on groups of 16 lanes: lane p of a group supplies the
// address of 4 columns at one k-row and receives 4 consecutive k of one column.  With
// p -> (k-row kb + p / 4, columns mb + 4 (p % 4)) lane p ends up with column mb + p, k = kb .. kb + 3; two reads
// (kb and kb + 4) give the 8 k of an MFMA operand.  A pass of 32 lanes (groups 0 and 1: 32 columns at 4 k-rows) reads
// eight 32-byte pieces; the column pair picks bit 1 of the chunk index, the k-row bits 2 and 3, so they are 8
// different positions modulo 256 bytes.  The 32-row block i of the wave's 128 rows adds 4 i to the chunk index, which
// the XOR does not commute with: one per-lane offset per block; kk adds 8192 bytes, the second read 2048.
__device__ __forceinline__ uint32_t transposed_frag_offset(int R0, int blk, int lane) {
    const int p = lane & 15, G = lane >> 4;
    const int m = R0 + blk * 32 + ((G & 1) << 4) + ((p & 3) << 2);
    const int kr = ((G >> 1) << 3) + (p >> 2);
    return (uint32_t)(kr * 512 + ((((m >> 3) ^ ((kr & 3) << 2))) << 4) + ((m & 7) << 1));
}

// per-lane LDS byte addresses of one operand's fragments in the CURRENT stage
template <int TR> struct FragBase {
    uint32_t b[4]; // row-major: one per kk; transposed: one per 32-row block
};

template <int TR> __device__ __forceinline__ void make_frag_base(FragBase<TR> &f, uint32_t tile_lds_addr, int R0, int lane) {
    if constexpr (TR == 0) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) f.b[kk] = tile_lds_addr + rowmajor_frag_offset(R0, kk, lane);
    } else {
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) f.b[blk] = tile_lds_addr + transposed_frag_offset(R0, blk, lane);
    }
}
template <int TR> __device__ __forceinline__ void flip_stage(FragBase<TR> &f) {
#pragma unroll
    for (int q = 0; q < 4; ++q) f.b[q] ^= (uint32_t)(STAGE_CHUNKS * 16);
}

// All fragment reads are inline assembly with an immediate offset: (1) after an LDS-DMA load the compiler guards every
// LDS read it cannot prove disjoint with s_waitcnt vmcnt(0), which would drain the load pipeline at each fragment;
// (2) it keeps address arithmetic out of the MFMA stream.  The compiler therefore does not know these reads are in
// flight: wait_frags() must precede their use.
template <int TR, int I, int KK> __device__ __forceinline__ u32x4 read_frag(const FragBase<TR> &f) {
    if constexpr (TR == 0) {
        u32x4 r;
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(f.b[KK]), "n"(I * 4096));
        return r;
    } else {
        u32x2 lo, hi;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(f.b[I]), "n"(KK * 8192));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(f.b[I]), "n"(KK * 8192 + 2048));
        u32x4 r = {lo[0], lo[1], hi[0], hi[1]};
        return r;
    }
}

struct Frags {
    u32x4 p[4], q[4];
};

// All LDS reads of this wave have returned; the fragments are tied to the statement so that no MFMA using them can be
// moved above it.
__device__ __forceinline__ void wait_frags(Frags &f) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(f.p[0]), "+v"(f.p[1]), "+v"(f.p[2]), "+v"(f.p[3]), "+v"(f.q[0]), "+v"(f.q[1]), "+v"(f.q[2]),
                   "+v"(f.q[3]));
}

template <int PTR, int QTR, int KK>
__device__ __forceinline__ void load_frags(Frags &f, const FragBase<PTR> &pb, const FragBase<QTR> &qb) {
    static_for<4>([&](auto I) {
        f.p[I.value] = read_frag<PTR, I.value, KK>(pb);
        f.q[I.value] = read_frag<QTR, I.value, KK>(qb);
    });
}

// The 16 MFMAs of one k16 sub-step on `cur` in pinned slots of MMA_GROUP MFMAs, each followed by its share of the other
// instructions: the 8 fragment reads of sub-step KK (of the stage pb/qb point at) into `nxt` during the first half of
// the sub-step, so that the second half covers their latency, and the 8 calls `hook(IC<0..7>)`, which the callers use
// to issue one LDS-DMA or index load each.  A wave issues in order, so anything not placed between MFMAs would leave the
// matrix pipe idle for as long as it takes to issue.  Pairs of MFMAs measured best in the kernels (single MFMAs 2-3 %
// slower, although an isolated instruction-mix benchmark prefers them).  NI < 4: only the first NI of the wave's four
// 32-wide Q blocks hold valid rows; the MFMAs and fragment reads of the others are left out.
constexpr int MMA_GROUP = 2;
template <typename T, int PTR, int QTR, int KK, int NI = 4, typename Hook>
__device__ __forceinline__ void mma_step(Frags &cur, Frags &nxt, const FragBase<PTR> &pb, const FragBase<QTR> &qb,
                                         f32x16 (&acc)[4][4], Hook hook) {
    wait_frags(cur); // issued at least 8 MFMAs ago
    constexpr int SLOTS = 16 / MMA_GROUP;
    static_for<SLOTS>([&](auto S) {
        constexpr int t = S.value;
        __builtin_amdgcn_sched_barrier(0);
        static_for<MMA_GROUP>([&](auto M) {
            // the 4 x 4 blocks in boustrophedon order: consecutive MFMAs differ in one operand only (measured 0 - 1 % faster
            // than row by row on the six GEMMs of the Mixtral-shaped layer; the sums are the same)
            constexpr int m = t * MMA_GROUP + M.value, j = m >> 2, i = (j & 1) ? 3 - (m & 3) : (m & 3);
            if constexpr (i < NI) acc[j][i] = Elem<T>::mfma(cur.p[j], cur.q[i], acc[j][i]);
        });
        __builtin_amdgcn_sched_barrier(0);
        // fragment reads: 8 (4 P, 4 Q) over the first SLOTS / 2 slots
        constexpr int RPS = 16 / SLOTS; // reads per slot of the first half
        if constexpr (t < SLOTS / 2) {
            static_for<RPS>([&](auto R) {
                constexpr int r = t * RPS + R.value, f = r >> 1;
                if constexpr ((r & 1) == 0) {
                    if constexpr (NI > 0) nxt.p[f] = read_frag<PTR, f, KK>(pb);
                } else {
                    if constexpr (f < NI) nxt.q[f] = read_frag<QTR, f, KK>(qb);
                }
            });
        }
        // hooks: 8 over all slots (two per slot for groups of 4, every other slot for single MFMAs)
        if constexpr (SLOTS == 4) {
            hook(IC<2 * t>{});
            hook(IC<2 * t + 1>{});
        } else if constexpr (SLOTS == 8) {
            hook(S);
        } else if constexpr ((t & 1) == 1) {
            hook(IC<t / 2>{});
        }
    });
    __builtin_amdgcn_sched_barrier(0);
}

struct NoHook {
    template <typename G> __device__ __forceinline__ void operator()(G) const {}
};

// Every LDS-DMA load of this wave has landed and its LDS reads have returned; then meet the other waves.  "memory"
// keeps the compiler from moving LDS accesses across it.
#define XMA_WAIT_LOADS_AND_BARRIER() asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory")
#define XMA_WAIT_ALL_LOADS() asm volatile("s_waitcnt vmcnt(0)" ::: "memory")

// ------------------------------------------------------------------------------------------------
// K loop by quadrants.  A wave's 128 x 128 corner is four quadrants of 64 x 64 (2 x 2 accumulator tiles); a K step of 64
// is four phases, one quadrant each over all 64 k: (Q0,P0) (Q0,P1) (Q1,P1) (Q1,P0), where Q0 / Q1 are the two 64-row
// halves of the wave's Q rows and P0 / P1 those of its P rows.  A half of an operand tile is read from LDS completely in
// one phase - P1 in the first, Q1 in the second, Q0 and P0 of the next step in the third and fourth - and its LDS is free
// from then on, while the other half of the same step is still to be read.  So the loads of step kt + 2 go out in two
// groups, {Q0, P0} in phases 1 and 2 and {P1, Q1} in phases 3 and 4 of step kt, each into the place that was read two
// phases before, and are needed five to six phases later: about one and a half K steps of lead from two LDS stages, where
// a loop that reads a step k16 by k16 frees a stage only when the step is over and gets half of that.
//
//   phase      multiplies    reads from LDS      loads (into the LDS just freed)
//   1          Q0 P0         P1(kt)              Q0(kt+2)
//   2          Q0 P1         Q1(kt)              P0(kt+2)
//   barrier B  all waves have read P1, Q1 of kt; {Q0, P0}(kt+1) have landed
//   3          Q1 P1         Q0(kt+1)            P1(kt+2)
//   4          Q1 P0         P0(kt+1)            Q1(kt+2)
//   barrier A  all waves have read Q0, P0 of kt+1; {P1, Q1}(kt+1) have landed
//
// Q0 and P0 of a tile's first step are read in front of the loop, so a barrier of their own stands there for the loads that
// phase 2 of that step puts into their place.  Loads, reads and waits are those of k_schedule.hpp, which is checked on the host.
//
// The fragments of a half are 8 x 4 registers; P0(kt+1) goes to the registers of P1(kt), so the two P sets change roles
// every step.  Sums run over k in the same order as in a k16 by k16 walk: results are bit-identical.
//
// Measured against the k16 by k16 walk (timing build, cycles per steady step; 2048 = the MFMAs back to back): 2375 -> 2224
// (x @ W^T, 8 experts of H = 4096, I = 14336, 16384 rows), 2594 -> 2266 (dy @ W, same), and the two or three steps behind a
// tile's first, which wait for panels that are not in L2 yet, 2800 - 4400 -> 2180 - 2300.  Launches 3 to 12 % shorter; the
// board's power limit takes back part of what the cycles give (the clock drops from 1.6 to 1.45 GHz).
//
// LDS layouts, 32 KB per operand tile as above.  Row-major: [256 rows][8 chunks], a wave loads rows
// half_row(wave, piece): 8 rows per LDS-DMA piece, four pieces per half.  Transposed source: two halves of
// [64 k-rows][16 chunks] (the 64-column groups 0, 2 and 1, 3 of the tile), chunk c of k-row kr at slot c ^ ((kr & 3) << 2):
// a piece covers four k-rows, two whole 128-byte lines each.
// ------------------------------------------------------------------------------------------------
struct Half {
    u32x4 f[4][2]; // [k16 step][32-row block]
};

// first of the 8 rows of row-major piece i (0..3: half 0, 4..7: half 1)
__device__ __forceinline__ int half_row(int wave, int i) { return (wave & 1) * 32 + (wave >> 1) * 128 + (i >> 2) * 64 + (i & 3) * 8; }
// transposed piece i: first of its 4 k-rows; the lane's k-row is + (lane >> 4)
__device__ __forceinline__ int half_krow(int wave, int i) { return wave * 16 + (i & 3) * 4; }
// the 16-byte column chunk (of the tile's 32) that this lane fetches for transposed piece i
__device__ __forceinline__ int half_col_chunk(int i, int lane) {
    const int c = (lane & 15) ^ (((lane >> 4) & 3) << 2);
    return (c >> 3) * 16 + (i >> 2) * 8 + (c & 7);
}
// LDS byte offset of piece i inside its operand tile
template <int TR> __device__ __forceinline__ int half_piece_lds(int wave, int i) {
    return TR == 0 ? half_row(wave, i) * 128 : (i >> 2) * 16384 + half_krow(wave, i) * 256;
}

template <int TR> struct HalfBase {
    uint32_t b[TR == 0 ? 4 : 2]; // row-major: one per k16 step; transposed: one per block of a half
};
template <int TR> __device__ __forceinline__ void make_half_base(HalfBase<TR> &f, uint32_t tile_lds_addr, int R0, int lane) {
    if constexpr (TR == 0) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) f.b[kk] = tile_lds_addr + rowmajor_frag_offset(R0, kk, lane);
    } else {
        const int p = lane & 15, G = lane >> 4;
        const int kr = ((G >> 1) << 3) + (p >> 2);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int c = (R0 >> 7) * 8 + b * 4 + ((G & 1) << 1) + ((p & 3) >> 1);
            f.b[b] = tile_lds_addr + (uint32_t)(kr * 256 + ((c ^ ((kr & 3) << 2)) << 4) + ((p & 1) << 3));
        }
    }
}
template <int TR> __device__ __forceinline__ void flip_half_base(HalfBase<TR> &f) {
#pragma unroll
    for (int q = 0; q < (TR == 0 ? 4 : 2); ++q) f.b[q] ^= (uint32_t)(STAGE_CHUNKS * 16);
}
template <int TR, int HALF, int KK, int B> __device__ __forceinline__ u32x4 read_half_frag(const HalfBase<TR> &f) {
    if constexpr (TR == 0) {
        u32x4 r;
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(f.b[KK]), "n"((HALF * 2 + B) * 4096));
        return r;
    } else {
        u32x2 lo, hi;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(f.b[B]), "n"(HALF * 16384 + KK * 4096));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(f.b[B]), "n"(HALF * 16384 + KK * 4096 + 1024));
        u32x4 r = {lo[0], lo[1], hi[0], hi[1]};
        return r;
    }
}
// the eight fragments tied to this point: no MFMA that uses them moves above it (the wait itself stands in front)
__device__ __forceinline__ void tie_half(Half &h) {
    asm volatile("" : "+v"(h.f[0][0]), "+v"(h.f[0][1]), "+v"(h.f[1][0]), "+v"(h.f[1][1]), "+v"(h.f[2][0]), "+v"(h.f[2][1]),
                      "+v"(h.f[3][0]), "+v"(h.f[3][1]));
}
#define XMA_WAIT_READS() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
// its LDS reads have returned (and all but the N youngest loads of this wave have landed); then meet the other waves
#define XMA_WAIT_READS_AND_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")
#define XMA_WAIT_AND_BARRIER(N) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory")

// The 16 MFMAs of a quadrant in eight slots of two.  Behind each slot: its share of the eight fragment reads (two, one,
// one, two, one, one: the LDS serves four waves, and the last read still has a slot and a half to return) and one call of
// the hook, which the callers use for a load every other slot.  NB < 2: only the first NB 32-row blocks of the Q half
// hold valid rows.
template <typename T, int J0, int I0, int NB, typename Read, typename Hook>
__device__ __forceinline__ void quadrant(const Half &p, const Half &q, f32x16 (&acc)[4][4], Read read, Hook hook) {
    static_for<8>([&](auto S) {
        constexpr int t = S.value;
        __builtin_amdgcn_sched_barrier(0);
        static_for<2>([&](auto M) {
            // (0,0) (0,1) (1,1) (1,0): consecutive MFMAs differ in one operand only
            constexpr int m = 2 * t + M.value, kk = m >> 2, j = (m >> 1) & 1, i = (m & 1) ^ j;
            if constexpr (i < NB) acc[J0 + j][I0 + i] = Elem<T>::mfma(p.f[kk][j], q.f[kk][i], acc[J0 + j][I0 + i]);
        });
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (t == 0) read(IC<0>{}), read(IC<1>{});
        if constexpr (t == 1) read(IC<2>{});
        if constexpr (t == 2) read(IC<3>{});
        if constexpr (t == 3) read(IC<4>{}), read(IC<5>{});
        if constexpr (t == 4) read(IC<6>{});
        if constexpr (t == 5) read(IC<7>{});
        hook(S);
    });
    __builtin_amdgcn_sched_barrier(0);
}
struct NoRead {
    template <typename R> __device__ __forceinline__ void operator()(R) const {}
};
template <int TR, int HALF, int NB> struct ReadHalf {
    Half &h;
    const HalfBase<TR> &base;
    template <typename R> __device__ __forceinline__ void operator()(R) const {
        constexpr int r = R::value, kk = r >> 1, b = r & 1;
        if constexpr (b < NB) h.f[kk][b] = read_half_frag<TR, HALF, kk, b>(base);
    }
};
template <int TR, int HALF, int NB> __device__ __forceinline__ ReadHalf<TR, HALF, NB> reader(Half &h, const HalfBase<TR> &base) {
    return ReadHalf<TR, HALF, NB>{h, base};
}

static_assert(4 * EPI_WAVE_BYTES <= GEMM_SMEM_BYTES && 4 * EPI_BWD_WAVE_BYTES <= GEMM_SMEM_BYTES,
              "epilogue staging must fit into the operand stages");

template <int N> __device__ __forceinline__ void zero_acc(f32x16 (&acc)[N][N]) {
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;
}

// The experts' bias enters a tile as a rank-one update of the cleared accumulators, ones (rows) x bias (columns), through
// the matrix pipe: one k16 step whose only non-zero k holds 1 in the Q fragments and the bias of the lane's column in the P
// fragments.  The product 1 x b is exact and it is the first term of the fp32 sum, so the result is rounded once, as a
// linear layer with a bias rounds it, and no epilogue has to know about the bias.  (Writing the bias into the
// accumulators directly, 256 register writes from loaded values, made the register allocation spill around the main loop.)
template <typename T>
__device__ __forceinline__ void add_bias(const FwdArgs &a, f32x16 (&acc)[4][4], int e, int n0, int wp, int lane) {
    const uint16_t *b = a.bias + (int64_t)e * a.bias_es;
    const bool k0 = lane < 32; // lanes 0..31 hold k = 0..7 of their row, lanes 32..63 k = 8..15
    u32x4 q = {k0 ? one_bits<T>() : 0u, 0u, 0u, 0u};
    u32x4 p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        int col = n0 + wp + 32 * j + (lane & 31);
        if (col >= a.N) col = a.N - 1; // columns past N are computed and never stored
        const uint32_t v = b[col];
        p[j] = u32x4{k0 ? v : 0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[j][i] = Elem<T>::mfma(p[j], q, acc[j][i]);
}

// The bias of this lane's four columns, zeros without one.  The values are used inside the branch, so that the wait for them
// stands there and covers loads that are older; behind it the compiler knows of no load to wait for.
struct Bias {
    uint32_t v[4];
};
__device__ __forceinline__ Bias load_bias(const FwdArgs &a, int e, int n0, int wp, int lane) {
    Bias r = {{0u, 0u, 0u, 0u}};
    if (a.bias != nullptr) { // uniform
        const uint16_t *b = a.bias + (int64_t)e * a.bias_es;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int col = n0 + wp + 32 * j + (lane & 31);
            if (col >= a.N) col = a.N - 1;
            r.v[j] = b[col];
        }
        asm volatile("" : "+v"(r.v[0]), "+v"(r.v[1]), "+v"(r.v[2]), "+v"(r.v[3]));
    }
    return r;
}

// The accumulators of a tile set to its expert's bias, or to zero without one, by MFMAs of that rank-one product onto a
// constant zero.  The blocks of a column block j have the same operands, so four MFMAs are left of the sixteen, and the first
// MFMA of each block reads one of their results as its addend: no register is written on its own.  The hook's loads are
// placed between them.
template <typename T, typename Hook>
__device__ __forceinline__ void init_acc(const Bias &bias, f32x16 (&acc)[4][4], int lane, Hook hook) {
    const bool k0 = lane < 32;
    const u32x4 q = {k0 ? one_bits<T>() : 0u, 0u, 0u, 0u};
    f32x16 zero;
#pragma unroll
    for (int c = 0; c < 16; ++c) zero[c] = 0.f;
    static_for<16>([&](auto S) {
        constexpr int j = S.value >> 2, i = S.value & 3;
        const u32x4 p = {k0 ? bias.v[j] : 0u, 0u, 0u, 0u};
        __builtin_amdgcn_sched_barrier(0);
        acc[j][i] = Elem<T>::mfma(p, q, zero);
        __builtin_amdgcn_sched_barrier(0);
        hook(S);
    });
}

// Which tile a workgroup works on.
struct TileSched {
    int e, rows_valid, n0; // expert, valid rows of the row tile, first output column
    int64_t row0;          // first grouped row
    int part, parts;       // K slice of a split tile (parts == 1: the whole K range)
    int tail_index;        // index of a split tile among the tiles of the last round
};

// Order of an expert's tiles.  The 32 consecutive tiles that xcd_remap hands to an XCD share operand panels in that XCD's
// L2: r row tiles x c column tiles need r activation panels and c weight panels for r c tiles, and the K loop runs as
// fast as those panels arrive.  Walking all row tiles of a column before the next column suits an expert of up to a
// dozen row tiles (measured best for 9: 9 + 3.6 panels, and the same activation panels in every round of the launch);
// an expert of 48 row tiles would have 32 tiles share one weight panel and fetch 32 activation panels (measured: the
// K loop of an expert of 64 row tiles takes 142 us instead of 100).  So the row tiles of a larger expert are cut into
// bands of equal height, at most FWD_BAND, and the walk goes down a band's column, then along the band, then to the next
// band.  Low bands measured better than square ones (4 x 8 before 6 x 5 before 8 x 4): a weight panel is one
// contiguous block, an activation panel 256 gathered rows.  local: index of the tile among the expert's tiles_m x NT.
constexpr int FWD_SINGLE_BAND_TILES = 12;
#ifdef XMA_PST_TIMING
__device__ int g_pst_band = 6; // A/B switch of the timing build
#define FWD_BAND g_pst_band
#else
constexpr int FWD_BAND = 6;
#endif
__device__ __forceinline__ void tile_of_expert(int local, int tiles_m, int NT, int &m_tile, int &n_tile) {
    if (tiles_m <= FWD_SINGLE_BAND_TILES) {
        m_tile = local % tiles_m, n_tile = local / tiles_m;
        return;
    }
    const int bands = (tiles_m + FWD_BAND - 1) / FWD_BAND;
    const int h = (tiles_m + bands - 1) / bands; // height of every band but the last, which has what is left
    int band = local / (h * NT);
    if (band > bands - 1) band = bands - 1;
    const int in_band = local - band * h * NT;
    const int rows = (band == bands - 1) ? tiles_m - h * (bands - 1) : h;
    m_tile = band * h + in_band % rows;
    n_tile = in_band / rows;
}

constexpr int SPLIT_MIN_STEPS = 8; // a K slice is at least this many K steps

// Expert-major schedule: work[e] = ceil(rows_e / BM) * n_tiles, prefix sum over the experts in LDS, then the tile of
// this workgroup.  With a workspace (a.partial) the tiles of the last, partial round of the launch - total mod
// split_cus of them, the workgroups that would otherwise run while most CUs idle - are cut into `parts` K slices, each
// taken by a workgroup of its own in a second launch of the kernel (ROLE_SLICES, at most split_cus workgroups); a
// third launch (ROLE_FIXUP, workgroup b = split tile b) adds the slices.  ROLE_TILES takes all other tiles.  Returns
// false if the workgroup has nothing to do.
constexpr int ROLE_TILES = 0, ROLE_SLICES = 1, ROLE_FIXUP = 2;
// grouped_gemm_kernel is the fallback of launch_fwd for launches that grouped_gemm_persistent_kernel does not take, and
// the kernel of the K slices.  Its SwiGLU-backward instantiations also walk several tiles per workgroup (one workgroup
// per compute unit), the others run one workgroup per tile.
__host__ __device__ constexpr bool fwd_persistent(int epi, int role) {
    return role == ROLE_TILES && epi_swiglu_bwd(epi);
}
template <int ROLE>
__device__ __forceinline__ bool locate_tile(const FwdArgs &a, unsigned char *smem, int *s_sched, TileSched &ts,
                                            int b, int tid) {
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NT = (a.N + BN - 1) / BN;
    int full = 0, rest = 0, parts = 1, part = 0, L = 0;
    // from the number of tiles: which one is this workgroup's (false: none)
    auto pick = [&](int total) -> bool {
        full = total;
        if (a.partial) {
            const int KT = (a.K + BK - 1) / BK;
            full = total / a.split_cus * a.split_cus;
            rest = total - full;
            parts = rest ? a.split_cus / rest : 1;
            if (parts > KT / SPLIT_MIN_STEPS) parts = KT / SPLIT_MIN_STEPS;
            if (parts < 2) parts = 1, full = total, rest = 0;
        }
        if (ROLE == ROLE_FIXUP) {
            if ((b >> 2) >= rest) return false; // four workgroups per split tile
            L = full + (b >> 2);
        } else if (ROLE == ROLE_SLICES) {
            if (rest == 0) return false;
            const int q = xcd_remap(b, a.split_cus); // neighbouring tiles of one slice index meet in one XCD's L2
            part = q / rest;
            if (part >= parts) return false;
            L = full + q % rest;
        } else {
            L = xcd_remap(b, a.grid_main);
            if (L >= full) return false; // beyond the last tile (the grid is an upper bound), or a tile that is split
        }
        return true;
    };
    int e, local;
    int64_t row_lo, row_hi;
    if (a.E <= WAVE) {
        // every wave scans the experts in registers: lane = expert; no LDS, no barrier, one load per lane
        const int64_t hi = a.offs[lane < a.E ? lane : a.E - 1];
        int64_t lo = __shfl_up(hi, 1);
        if (lane == 0) lo = 0;
        const int v = (int)((hi - lo + BM - 1) / BM) * NT; // 0 for the lanes past E
        int s = v;
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const int t = __shfl_up(s, d);
            if (lane >= d) s += t;
        }
        if (!pick(__builtin_amdgcn_readlane(s, WAVE - 1))) return false;
        const uint64_t hit = __ballot(s - v <= L && L < s); // exactly one lane
        e = __builtin_ctzll(hit);
        local = L - __builtin_amdgcn_readlane(s - v, e);
        row_lo = ((int64_t)__builtin_amdgcn_readlane((int)(lo >> 32), e) << 32) |
                 (uint32_t)__builtin_amdgcn_readlane((int)lo, e);
        row_hi = ((int64_t)__builtin_amdgcn_readlane((int)(hi >> 32), e) << 32) |
                 (uint32_t)__builtin_amdgcn_readlane((int)hi, e);
    } else {
        int *s_pre = (int *)smem; // [E + 1], dead before the first tile load
        if (wave == 0) {
            int carry = 0;
            for (int b = 0; b < a.E; b += WAVE) {
                const int x = b + lane;
                int v = 0;
                if (x < a.E) {
                    const int64_t cnt = a.offs[x] - (x ? a.offs[x - 1] : 0);
                    v = (int)((cnt + BM - 1) / BM) * NT;
                }
                int s = v;
#pragma unroll
                for (int d = 1; d < WAVE; d <<= 1) {
                    const int t = __shfl_up(s, d);
                    if (lane >= d) s += t;
                }
                if (x < a.E) s_pre[x] = carry + s - v;
                carry += __shfl(s, WAVE - 1);
            }
            if (lane == 0) s_pre[a.E] = carry;
        }
        __syncthreads();
        if (!pick(__builtin_amdgcn_readfirstlane(s_pre[a.E]))) return false;
        for (int x = tid; x < a.E; x += GEMM_THREADS)
            if (s_pre[x] <= L && L < s_pre[x + 1]) {
                s_sched[0] = x;
                s_sched[1] = L - s_pre[x];
            }
        __syncthreads();
        e = __builtin_amdgcn_readfirstlane(s_sched[0]);
        local = __builtin_amdgcn_readfirstlane(s_sched[1]);
        row_lo = e ? a.offs[e - 1] : 0;
        row_hi = a.offs[e];
        __syncthreads(); // s_pre is dead from here on
    }
    const int tiles_m = (int)((row_hi - row_lo + BM - 1) / BM);
    int m_tile, n_tile;
    tile_of_expert(local, tiles_m, NT, m_tile, n_tile);
    ts.e = e;
    ts.row0 = row_lo + (int64_t)m_tile * BM;
    ts.rows_valid = (int)((row_hi - ts.row0 < BM) ? row_hi - ts.row0 : BM);
    ts.n0 = n_tile * BN;
    ts.part = part;
    ts.parts = (L >= full) ? parts : 1;
    ts.tail_index = L - full;
    return true;
}

// ------------------------------------------------------------------------------------------------
// forward / dX kernel
//   WT = 0: W[e] is (N, K) with K contiguous (x @ W^T)      -> P tile row-major
//   WT = 1: W[e] is (K, N) with N contiguous (dy @ W)       -> P tile transposed source
// ------------------------------------------------------------------------------------------------
template <typename T, int WT, int EPI, int ROLE>
__global__ __launch_bounds__(GEMM_THREADS, 1) void grouped_gemm_kernel(const FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int s_sched[4];
    u32x4 *tiles = (u32x4 *)smem;
    // A persistent launch has one workgroup per compute unit, which walks the tiles b, b + gridDim.x, ... of the launch.
    const int b_end = fwd_persistent(EPI, ROLE) ? a.grid_main : (int)blockIdx.x + 1;
    for (int b = blockIdx.x; b < b_end; b += gridDim.x) {
    if (b != (int)blockIdx.x) __syncthreads(); // the staging areas of the last epilogue are dead in every wave
    // Everything derived from the thread index is derived again for every tile (the compiler cannot see through the
    // empty statement): hoisted out of the tile loop, those values would live across the main loop, which has no
    // register to spare, and be spilled.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    TileSched ts;
    if (!locate_tile<ROLE>(a, smem, s_sched, ts, b, tid)) continue;
    const int e = ts.e, rows_valid = ts.rows_valid, n0 = ts.n0;
    const int64_t row0 = ts.row0;

    // ---- loader set-up: one fixed per-lane global pointer per LDS-DMA piece (k = 0); a step adds a uniform offset
    const uint16_t *zero = (const uint16_t *)g_zero_page;
    const int KT = (a.K + BK - 1) / BK;
    const bool k_tail = (a.K & (BK - 1)) != 0; // the last step has chunks past K: they are fetched from the zero page
    // K steps [kt0, kt1) of this workgroup: all of them, or one of ts.parts slices of a tile of the last round.  kt0 is
    // even, so step kt lives in stage kt & 1 in either case.
    const int kt0 = (ROLE == ROLE_SLICES) ? ((ts.part * KT / ts.parts) & ~1) : 0;
    const int kt1 = (ROLE == ROLE_SLICES && ts.part + 1 < ts.parts) ? (((ts.part + 1) * KT / ts.parts) & ~1) : KT;
    const uint16_t *q_ptr[8], *p_ptr[8];
    {
        const uint16_t *We = a.W + (int64_t)e * a.w_es;
        if (WT == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                int r = n0 + wave * 64 + i * 8 + (lane >> 3);
                if (r >= a.N) r = a.N - 1;
                p_ptr[i] = We + (int64_t)r * a.ldw + rowmajor_lane_chunk(i, lane) * 8;
            }
        } else {
            const int max_chunk = ((a.N - n0) >> 3) - 1; // last valid 16-byte chunk of the tile's column range
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                int cj = transposed_lane_chunk(j, lane);
                if (cj > max_chunk) cj = max_chunk; // columns past the edge are masked at the store
                p_ptr[j] = We + (int64_t)(wave * 16 + 2 * j + (lane >> 5)) * a.ldw + n0 + cj * 8;
            }
        }
    }
    const int64_t p_step = (WT == 0) ? BK : (int64_t)BK * a.ldw; // elements per K step along the P pointers
    const uint32_t lds0 = lds_addr_of(smem);

    // piece 0..15 of K step kt -> stage kt & 1 (pieces 0..7 = Q tile, 8..15 = P tile).  FULL: the caller guarantees
    // that step kt exists and has no chunk past K, so the piece is one M0 update, one 64-bit add and the load; a wave
    // with a single instruction stream cannot afford more than a few instructions per MFMA.
    auto issue_piece = [&](int kt, auto PIECE, auto FULL) {
        constexpr int piece = PIECE.value;
        constexpr int slot =
            (piece >> 3) * OP_CHUNKS + ((piece < 8 || WT == 0) ? (piece & 7) * 64 : (piece & 7) * 64); // 1 KB per piece
        if constexpr (!FULL.value) {
            if (kt >= kt1) return; // uniform
        }
        u32x4 *dst = tiles + (kt & 1) * STAGE_CHUNKS + slot + wave * 512; // a wave's 8 pieces are 8 KB apart per wave
        const uint16_t *src;
        if constexpr (piece < 8)
            src = q_ptr[piece] + (int64_t)kt * BK;
        else
            src = p_ptr[piece - 8] + (int64_t)kt * p_step;
        if constexpr (!FULL.value) {
            if (k_tail && kt == KT - 1) { // uniform branch, taken by at most one step of a tile
                asm volatile("" ::: "memory"); // keeps this rare path a branch instead of selects in every piece
                if (piece < 8 || WT == 0) {
                    if (kt * BK + rowmajor_lane_chunk(piece & 7, lane) * 8 >= a.K) src = zero;
                } else {
                    if (kt * BK + wave * 16 + 2 * (piece - 8) + (lane >> 5) >= a.K) src = zero;
                }
            }
        }
        lds_dma16(src, dst);
    };

    f32x16 acc[4][4];
    zero_acc(acc);
    const int wq = (wave & 1) * 128, wp = (wave >> 1) * 128; // wave's 128 x 128 corner inside the tile
    if (a.bias != nullptr && kt0 == 0) add_bias<T>(a, acc, e, n0, wp, lane); // the first K slice of a split tile only
    FragBase<0> qb;
    FragBase<WT> pb;
    make_frag_base<0>(qb, lds0, wq, lane);
    make_frag_base<WT>(pb, lds0 + OP_CHUNKS * 16, wp, lane);

    // The weight pieces of the first step go out before the activation rows are known: their addresses need only
    // the schedule, while the rows of a gathered tile take another dependent load (the scattered index).
    static_for<8>([&](auto P) { issue_piece(kt0, IC<8 + P.value>{}, IC<0>{}); });
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        int r = wave * 64 + i * 8 + (lane >> 3);
        if (r >= rows_valid) r = rows_valid - 1; // duplicates, masked at the store
        const int64_t n = row0 + r;
        const int64_t src = a.x_grouped ? n : (int64_t)fastdiv((uint32_t)a.idx[n], a.fan_div);
        q_ptr[i] = a.X + src * a.ldx + rowmajor_lane_chunk(i, lane) * 8;
    }
    static_for<8>([&](auto P) { issue_piece(kt0, P, IC<0>{}); });
    static_for<DMA_N0>([&](auto P) { issue_piece(kt0 + 1, P, IC<0>{}); });
    // the first step has landed in every wave (the first loads of the second may be in flight)
    if (kt1 - kt0 > 1)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(DMA_N0) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    // Q blocks (32 rows) of this wave that hold valid rows: 4 except in an expert's last row tile.  A wave with fewer
    // skips the MFMAs and fragment reads of the empty blocks (rounded up to 0, 1, 2 or 4 blocks); it still issues its
    // share of the loads and meets every barrier.
    const int q_blocks = (rows_valid > wq) ? (rows_valid - wq + 31) >> 5 : 0;
    const int KT_full = (a.K / BK < kt1) ? a.K / BK : kt1; // end of the steps without a chunk past K
    auto main_loop = [&](auto NI_) {
        constexpr int NI = NI_.value;
        Frags f0, f1;
        if constexpr (NI > 0) {
            static_for<4>([&](auto I) { f0.p[I.value] = read_frag<WT, I.value, 0>(pb); });
            static_for<NI>([&](auto I) { f0.q[I.value] = read_frag<0, I.value, 0>(qb); });
        }
        // one K step; FULL: steps kt + 1 and kt + 2 exist and are complete
        auto k_step = [&](int kt, auto FULL) {
            // The step numbers of the loads are made opaque: otherwise the compiler turns "pointer + kt * step" into 16
            // running pointers and advances all of them with 64-bit vector adds in one lump at the end of the loop body,
            // where nothing hides them.
            int kt_a = kt + 1, kt_b = kt + 2;
            asm volatile("" : "+s"(kt_a), "+s"(kt_b));
            // rest of the loads of step kt + 1 (the first DMA_N0 went out behind the previous barrier)
            mma_step<T, WT, 0, 1, NI>(f0, f1, pb, qb, acc, [&](auto G) {
                if constexpr (G.value < DMA_N1) issue_piece(kt_a, IC<DMA_N0 + G.value>{}, FULL);
            });
            mma_step<T, WT, 0, 2, NI>(f1, f0, pb, qb, acc, [&](auto G) {
                if constexpr (G.value < DMA_N2) issue_piece(kt_a, IC<DMA_N0 + DMA_N1 + G.value>{}, FULL);
            });
            mma_step<T, WT, 0, 3, NI>(f0, f1, pb, qb, acc, NoHook());
            XMA_WAIT_LOADS_AND_BARRIER(); // step kt + 1 has landed; nobody reads this stage any more
            flip_stage(pb);
            flip_stage(qb);
            // the stage just left is free: first loads of step kt + 2; fragments of sub-step 0 of step kt + 1
            mma_step<T, WT, 0, 0, NI>(f1, f0, pb, qb, acc, [&](auto G) {
                if constexpr (G.value < DMA_N0) issue_piece(kt_b, G, FULL);
                if constexpr (G.value + 8 < DMA_N0) issue_piece(kt_b, IC<G.value + 8>{}, FULL);
            });
        };
        int kt = kt0;
        if constexpr (NI == 4)
            for (; kt + 2 < KT_full; ++kt) k_step(kt, IC<1>{});
        for (; kt < kt1; ++kt) k_step(kt, IC<0>{});
        // The last sub-step reads ahead for a step that does not exist.  Nobody uses these fragments, so the compiler would
        // take their registers, to move the accumulators where the four loops meet, while the reads are in flight.
        wait_frags(f0);
    };
    if (q_blocks > 2)
        main_loop(IC<4>{});
    else if (q_blocks == 2)
        main_loop(IC<2>{});
    else if (q_blocks == 1)
        main_loop(IC<1>{});
    else
        main_loop(IC<0>{});
    // every load has landed, every fragment read has returned, and no wave touches the operand tiles any more: LDS becomes
    // the staging area of the epilogue
    XMA_WAIT_LOADS_AND_BARRIER();

    if constexpr (ROLE == ROLE_SLICES) {
        // one K slice of a tile of the last round: the fp32 accumulators go to the workspace, 16 bytes per lane and
        // consecutive lanes side by side; grouped_gemm_fixup_kernel adds the slices and runs the epilogue
        float4 *dst = (float4 *)a.partial + (size_t)(ts.tail_index * ts.parts + ts.part) * (BM * BN / 4) + tid;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    dst[((j * 4 + i) * 4 + g) * GEMM_THREADS] =
                        make_float4(acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]);
    } else {
        int tid_e = threadIdx.x;
        asm volatile("" : "+v"(tid_e));
        tile_epilogue<T, EPI>(a, acc, smem, row0, rows_valid, n0, tid_e);
    }
    }
}

// Sum of the K slices of the split tiles of the last round, then the epilogue of the GEMM kernel.  Four workgroups
// per split tile, one per 32-row block of the waves' corners (a quarter of the loads each: the kernel is a chain of
// dependent round trips, so it is as fast as it is parallel); the slices are added in a fixed order, so the result does
// not depend on timing.
template <typename T, int EPI>
__global__ __launch_bounds__(GEMM_THREADS, 1) void grouped_gemm_fixup_kernel(const FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int s_sched[4];
    TileSched ts;
    if (!locate_tile<ROLE_FIXUP>(a, smem, s_sched, ts, (int)blockIdx.x, (int)threadIdx.x)) return;
    const int tid = threadIdx.x;
    const int iblk = blockIdx.x & 3;
    f32x16 acc[4][4];
    zero_acc(acc);
    for (int p = 0; p < ts.parts; ++p) {
        const float4 *src = (const float4 *)a.partial + (size_t)(ts.tail_index * ts.parts + p) * (BM * BN / 4) + tid;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i != iblk) continue;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 v = src[((j * 4 + i) * 4 + g) * GEMM_THREADS];
                    acc[j][i][4 * g] += v.x, acc[j][i][4 * g + 1] += v.y, acc[j][i][4 * g + 2] += v.z, acc[j][i][4 * g + 3] += v.w;
                }
            }
    }
    tile_epilogue<T, EPI>(a, acc, smem, ts.row0, ts.rows_valid, ts.n0, (int)threadIdx.x, iblk);
}

// ------------------------------------------------------------------------------------------------
// Persistent forward / dX kernel: one workgroup per compute unit walks the tiles b, b + gridDim.x, ... of the launch and
// overlaps the set-up of a tile with the epilogue of the tile before it.
//
// Between two main loops a workgroup has to find its next tile, fetch the scattered row indices, and wait for the first
// K step to arrive from HBM: three dependent round trips with idle matrix pipes, as long as the epilogue itself.  Here
// everything a tile needs is fetched one tile ahead: while tile i is in its main loop the entry of tile i + 1 is read from
// the table of the workgroup's tiles and its row indices go into LDS, and the 16 LDS-DMA pieces of its first K step go out
// in the last step of tile i or right behind its main loop, before its epilogue starts.  They land
// in stage 0 while the epilogue stages its rows in the LDS above it (stage 1 and the 32 KB that the two stages leave
// free), so the next main loop starts as soon as the epilogue's stores have been handed over.
//
// The LDS-DMA loads are issued from inline assembly here (M0 is written next to the load): the compiler guards every
// LDS access it cannot prove disjoint from an LDS-DMA load it knows of with s_waitcnt vmcnt(0), which would make the
// epilogue wait for the loads it is supposed to hide.  What the compiler does not know it cannot wait for too little
// either: vmcnt retires in order, so a wait sized for the compiler's own loads only ever covers more than it has to; the
// waits that protect the operand tiles are all explicit.
//
// The expert-major schedule (tiles before each expert, row offsets) is computed once per workgroup into LDS instead of
// once per tile.  E <= PST_MAX_E; launches with more experts use grouped_gemm_kernel.
// ------------------------------------------------------------------------------------------------
constexpr int PST_MAX_E = 1023;
constexpr int PST_SMEM_BYTES = 160 * 1024 - 64;
constexpr int PST_STAGING_OFF = STAGE_CHUNKS * 16; // the epilogue's staging area starts above stage 0
// Rows fetched one tile ahead wait in LDS, one dword per row and wave, so that no register is held across the main loop.
// An item is 64 rows of each wave (1 KB): one of gathered rows of the next tile, 2 x 2 of rows of the epilogue (the next
// tile's arrive while this tile's are still needed), two of row scales of this tile.
constexpr int PST_ROWS_OFF = PST_STAGING_OFF + 4 * EPI_BWD_WAVE_BYTES;
constexpr int PST_QR = 0, PST_ER = 1, PST_SC = 5, PST_ROW_ITEMS = 7;
constexpr int PST_TABLE_OFF = PST_SMEM_BYTES - 2 * (PST_MAX_E + 1) * (int)sizeof(int);
constexpr int PST_WALK = GEMM_THREADS, PST_WALK_OFF = PST_TABLE_OFF - PST_WALK * 16 - 16; // entries; counts of the waves behind them
constexpr int PST_STEP_LDS_OFF = PST_ROWS_OFF + PST_ROW_ITEMS * 1024; // timing build: 8 bytes per K step, up to the tables
static_assert(EPI_BWD_WAVE_BYTES >= EPI_WAVE_BYTES && PST_ROWS_OFF + PST_ROW_ITEMS * 1024 <= PST_WALK_OFF,
              "epilogue staging and the prefetched rows must fit between stage 0 and the schedule tables");

__device__ __forceinline__ void lds_dma16_raw(const void *src, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_wave_base), "v"(src)
                 : "memory", "m0");
}
// one dword per lane: lane l's value lands at lds_wave_base + 4 l
__device__ __forceinline__ void lds_dma4_raw(const void *src, uint32_t lds_wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_wave_base), "v"(src)
                 : "memory", "m0");
}

// the same through a buffer descriptor
__device__ __forceinline__ void lds_dma4_buf(i32x4 desc, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_base), "v"(off), "s"(desc)
                 : "memory", "m0");
}
// Optional phase stamps of the persistent kernel (builds with -DXMA_PST_TIMING only): workgroup b writes the 100 MHz
// real-time counter at six points of each of its first PST_TIMING_TILES tiles; xma_rocm_debug_pst_times copies them out.
#ifdef XMA_PST_TIMING
constexpr int PST_TIMING_TILES = 48;
__device__ uint64_t g_pst_times[256][PST_TIMING_TILES][8];
__device__ uint64_t g_pst_cycles[256][PST_TIMING_TILES][8]; // the shader clock counter at the same points
__device__ int g_pst_no_ovl; // A/B switch of the timing build: 1 = no tile overlaps its neighbours' set-up
// the shader clock counter behind every K step of one tile per workgroup (the PST_STEP_TILE-th): written to a spare
// corner of LDS inside the loop (a vector store to memory would enter the loop's vmcnt waits), copied out behind the tile
constexpr int PST_STEP_TILE = 3, PST_MAX_STEPS = 240;
__device__ uint64_t g_pst_steps[256][PST_MAX_STEPS];
#define PST_STEP_STAMP(kt)                                                                             \
    do {                                                                                               \
        if (tile_no == PST_STEP_TILE && threadIdx.x == 0 && (kt) < PST_MAX_STEPS)                      \
            ((uint64_t *)(smem + PST_STEP_LDS_OFF))[(kt)] = __builtin_amdgcn_s_memtime();             \
    } while (0)
#define PST_STAMP(k)                                                                                   \
    do {                                                                                               \
        if (threadIdx.x == 0 && blockIdx.x < 256 && tile_no < PST_TIMING_TILES) {                      \
            g_pst_times[blockIdx.x][tile_no][k] = __builtin_amdgcn_s_memrealtime();                    \
            g_pst_cycles[blockIdx.x][tile_no][k] = __builtin_amdgcn_s_memtime();                       \
        }                                                                                              \
    } while (0)
#else
#define PST_STAMP(k) \
    do {             \
    } while (0)
#define PST_STEP_STAMP(kt) \
    do {                   \
    } while (0)
#endif

struct PstTile {
    int valid, n, e, n0, rows_valid, row0; // n: index in the table of the workgroup's walk
};

template <typename T, int WT, int EPI>
__global__ __launch_bounds__(GEMM_THREADS, 1) void grouped_gemm_persistent_kernel(const FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    int *s_pre = (int *)(smem + PST_TABLE_OFF); // [E + 1] tiles of the experts before e
    int *s_hi = s_pre + (PST_MAX_E + 1);        // [E] inclusive row offsets
    const int NT = (a.N + BN - 1) / BN;
    const int KT = (a.K + BK - 1) / BK;
    const bool k_tail = (a.K & (BK - 1)) != 0;
    const uint32_t lds0 = lds_addr_of(smem);

    // ---- schedule tables, once per workgroup
    {
        const int tid0 = threadIdx.x, lane0 = tid0 & 63;
        if (tid0 < WAVE) {
            int carry = 0;
            for (int b = 0; b < a.E; b += WAVE) {
                const int x = b + lane0;
                int v = 0;
                if (x < a.E) {
                    const int64_t hi = a.offs[x];
                    const int64_t cnt = hi - (x ? a.offs[x - 1] : 0);
                    v = (int)((cnt + BM - 1) / BM) * NT;
                    s_hi[x] = (int)hi;
                }
                int s = v;
#pragma unroll
                for (int d = 1; d < WAVE; d <<= 1) {
                    const int t = __shfl_up(s, d);
                    if (lane0 >= d) s += t;
                }
                if (x < a.E) s_pre[x] = carry + s - v;
                carry += __shfl(s, WAVE - 1);
            }
            if (lane0 == 0) s_pre[a.E] = carry;
        }
        __syncthreads();
    }
    int full = __builtin_amdgcn_readfirstlane(s_pre[a.E]); // tiles this launch computes whole
    if (a.partial) { // the tiles of a last, partial round are left to the K-slice and fix-up launches (see locate_tile)
        const int total = full;
        full = total / a.split_cus * a.split_cus;
        const int rest = total - full;
        int parts = rest ? a.split_cus / rest : 1;
        if (parts > KT / SPLIT_MIN_STEPS) parts = KT / SPLIT_MIN_STEPS;
        if (parts < 2) full = total;
    }

    // The workgroup's walk: the tiles blockIdx.x + i * gridDim.x of the launch that exist, PST_WALK of them at a time as
    // table entries in LDS (expert, first column, valid rows, first row), found by one binary search per thread.  The next
    // tile of the walk is then one 16-byte LDS read, which the main loop of the tile before it can afford anywhere.
    i32x4 *s_walk = (i32x4 *)(smem + PST_WALK_OFF);
    int *s_cnt = (int *)(s_walk + PST_WALK);
    int walk_pos = 0; // candidates i looked at so far
    // fills the table from candidate walk_pos on; returns the number of entries (0: the walk is over).  All waves meet here.
    auto fill_walk = [&](int tid) -> int {
        const int lane = tid & 63, wave = tid >> 6;
        for (;;) {
            const int64_t t = (int64_t)blockIdx.x + (int64_t)(walk_pos + tid) * gridDim.x;
            if ((int64_t)blockIdx.x + (int64_t)walk_pos * gridDim.x >= a.grid_main) return 0;
            const int L = t < a.grid_main ? xcd_remap((int)t, a.grid_main) : full;
            const uint64_t have = __ballot(L < full);
            if (lane == 0) s_cnt[wave] = __popcll(have);
            __syncthreads();
            int before = __popcll(have & ((1ull << lane) - 1)), total = 0;
            for (int w = 0; w < 4; ++w) {
                if (w < wave) before += s_cnt[w];
                total += s_cnt[w];
            }
            if (L < full) {
                int lo = 0, hi = a.E; // s_pre[lo] <= L < s_pre[hi]
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (s_pre[mid] <= L)
                        lo = mid;
                    else
                        hi = mid;
                }
                const int row_hi = s_hi[lo], row_lo = lo ? s_hi[lo - 1] : 0;
                int m_tile, n_tile;
                tile_of_expert(L - s_pre[lo], (row_hi - row_lo + BM - 1) / BM, NT, m_tile, n_tile);
                const int row0 = row_lo + m_tile * BM;
                s_walk[before] = i32x4{lo, n_tile * BN, (row_hi - row0 < BM) ? row_hi - row0 : BM, row0};
            }
            __syncthreads();
            walk_pos += PST_WALK;
            if (total) return __builtin_amdgcn_readfirstlane(total);
        }
    };
    int walk_len = 0; // entries of the table
    auto entry = [&](int n) -> PstTile {
        const i32x4 w = s_walk[n < walk_len ? n : 0];
        PstTile r;
        r.valid = __builtin_amdgcn_readfirstlane(n < walk_len ? 1 : 0);
        r.n = n;
        r.e = __builtin_amdgcn_readfirstlane(w[0]);
        r.n0 = __builtin_amdgcn_readfirstlane(w[1]);
        r.rows_valid = __builtin_amdgcn_readfirstlane(w[2]);
        r.row0 = __builtin_amdgcn_readfirstlane(w[3]);
        return r;
    };
    // Rows of a wave whose scattered indices are needed: the 64 rows of its LDS-DMA pieces (one item: lane l holds row
    // l % 8 of piece l / 8) and the 128 rows of its epilogue (two items: lane l of item m holds row 64 m + l), clamped to
    // the tile's last valid row (duplicates are computed and never stored).  An item is one 4-byte LDS-DMA load (the low
    // dword of the index) into the wave's part of the row area.
    const uint32_t *idx32 = (const uint32_t *)a.idx;
    const bool need_q_idx = !a.x_grouped, need_e_idx = !a.y_grouped || a.scale != nullptr;
    auto clamp_row = [&](const PstTile &t, int r) { return r < t.rows_valid ? r : t.rows_valid - 1; };
    auto row_item_lds = [&](int item, int wave) { return lds0 + (uint32_t)(PST_ROWS_OFF + item * 1024 + wave * 256); };
    auto row_item = [&](int item, int wave, int slot) {
        return ((const uint32_t *)(smem + PST_ROWS_OFF + item * 1024 + wave * 256))[slot];
    };
    // The five items of a tile's main loop: 0 the gathered rows of the next tile, 1, 2 the rows of its epilogue, 3, 4 the
    // row scales of this tile (the aligned dword that holds the 16-bit scale; the host checks that the vector starts on 4
    // bytes).  One that is not needed is a load from an empty buffer, so that their number is always five.
    constexpr int ROW_LOADS = k_schedule::ROW_LOADS;
    auto prefetch_item = [&](auto ITEM, const PstTile &t, int lane, int wave, int e_buf) {
        constexpr int it = ITEM.value;
        if constexpr (it < 3) {
            const bool need = t.valid && (it == 0 ? need_q_idx : need_e_idx);
            const int r = clamp_row(t, it == 0 ? half_row(wave, 0) + (lane >> 5) * 64 + (lane & 31) : (wave & 1) * 128 + (it - 1) * 64 + lane);
            lds_dma4_buf(buf_desc(idx32 + 2 * (int64_t)t.row0, need ? 0xfffffff0u : 0u), (uint32_t)r * 8,
                         row_item_lds(it == 0 ? PST_QR : PST_ER + 2 * (e_buf ^ 1) + (it - 1), wave));
        } else {
            const uint32_t s_idx = row_item(PST_ER + 2 * e_buf + (it - 3), wave, lane);
            lds_dma4_buf(buf_desc(a.scale, a.scale ? 0xfffffff0u : 0u), (s_idx >> 1) * 4, row_item_lds(PST_SC + (it - 3), wave));
        }
    };

    // Addresses of the 16 LDS-DMA pieces of a tile (0..3 Q0, 4..7 Q1, 8..11 P0, 12..15 P1): a uniform base per operand
    // (SGPRs: the tile's corner of the weight matrix; the activations' first row for a gathered operand, the tile's first
    // row for a grouped one) and one 32-bit byte offset per piece and lane.  A K step adds a uniform amount to the bases,
    // so a piece in the loop is the M0 update and the load, without any vector address arithmetic.  The host has checked
    // that the offsets fit 32 bits.
    uint32_t q_off[8], p_off[8];
    const char *q_base = nullptr, *p_base = nullptr;
    uint32_t tile_bytes = 0xfffffff0u; // size in the buffer descriptors: 0 for a tile that does not exist
    const int64_t p_step_b = (WT == 0) ? 2 * BK : (int64_t)2 * BK * a.ldw; // bytes per K step along the weights
    auto make_bases = [&](const PstTile &t) {
        const uint16_t *We = a.W + (int64_t)t.e * a.w_es;
        p_base = (WT == 0) ? (const char *)(We + (int64_t)t.n0 * a.ldw) : (const char *)(We + t.n0);
        q_base = (const char *)(need_q_idx ? a.X : a.X + (int64_t)t.row0 * a.ldx);
        tile_bytes = t.valid ? 0xfffffff0u : 0u;
    };
    auto make_p_off = [&](const PstTile &t, auto I_, int lane, int wave) {
        constexpr int i = I_.value;
        if (WT == 0) {
            int r = half_row(wave, i) + (lane >> 3);
            if (t.n0 + r >= a.N) r = a.N - 1 - t.n0;
            p_off[i] = mul_add_u32((uint32_t)r, (uint32_t)(2 * a.ldw), (uint32_t)rowmajor_lane_chunk(i, lane) * 16);
        } else {
            const int max_chunk = ((a.N - t.n0) >> 3) - 1;
            int cj = half_col_chunk(i, lane);
            if (cj > max_chunk) cj = max_chunk;
            p_off[i] = mul_add_u32((uint32_t)(half_krow(wave, i) + (lane >> 4)), (uint32_t)(2 * a.ldw), (uint32_t)cj * 16);
        }
    };
    // The row of piece i of a lane is the scattered index that the row item holds, divided by fan_out, for a gathered operand
    // and the row inside the tile for a grouped one (where the launch has set the divisor to one).
    const uint32_t gather_mask = need_q_idx ? 0xffffffffu : 0u;
    auto make_q_off = [&](const PstTile &t, auto I_, int lane, int wave, uint32_t idx) {
        constexpr int i = I_.value;
        const uint32_t local = (uint32_t)clamp_row(t, half_row(wave, i) + (lane >> 3));
        const uint32_t src = fastdiv((idx & gather_mask) | (local & ~gather_mask), a.fan_div);
        q_off[i] = mul_add_u32(src, (uint32_t)(2 * a.ldx), (uint32_t)rowmajor_lane_chunk(i, lane) * 16);
    };
    int wave_u = 0; // this wave's index, set per tile (uniform)
    int lane_v = 0;
    // one piece of K step kt of the tile the bases and offsets describe -> stage kt & 1.  FULL: the step exists and has no
    // chunk past K; otherwise every lane whose chunk lies past K (all of them in a step past the last one) asks for an
    // address outside the buffer, which the load answers with zeros, so that every step of a tile issues the same number
    // of loads: the waits count on that
    auto issue_piece = [&](int kt, auto PIECE, auto FULL) {
        constexpr int piece = PIECE.value;
        constexpr int tr = (piece < 8) ? 0 : WT;
        // LDS destination = the piece's place in stage 0 (loop invariant) + the stage; both uniform
        const uint32_t dst0 = lds0 + (uint32_t)((piece >> 3) * OP_CHUNKS * 16 + half_piece_lds<tr>(wave_u, piece & 7));
        const uint32_t stage = (uint32_t)((kt & 1) * STAGE_CHUNKS * 16);
        const char *base = (piece < 8) ? q_base + (int64_t)kt * (2 * BK) : p_base + (int64_t)kt * p_step_b; // uniform
        uint32_t off = (piece < 8) ? q_off[piece & 7] : p_off[piece & 7];
        if constexpr (!FULL.value) {
            const int k = (tr == 0) ? rowmajor_lane_chunk(piece & 7, lane_v) * 8 : half_krow(wave_u, piece & 7) + (lane_v >> 4);
            off = (k < a.K - kt * BK) ? off : BUF_OUTSIDE;
        }
        lds_dma16_buf(buf_desc(base, tile_bytes), off, dst0, stage);
    };
    auto ordered = [](auto P) { return IC<k_schedule::ordered(P.value)>{}; };

    // From here on the offsets are those of the last K step of a tile that overlaps: chunks past K lie outside the buffers.
    // (The loads of such a tile do not check; the next tile's offsets are made in that step.)
    auto cut_tail = [&]() {
        if (!k_tail) return;
        const int k_left = a.K - (KT - 1) * BK;
        static_for<8>([&](auto I) {
            constexpr int i = I.value;
            const bool in_row = rowmajor_lane_chunk(i, lane_v) * 8 < k_left;
            q_off[i] = in_row ? q_off[i] : BUF_OUTSIDE;
            p_off[i] = (WT == 0 ? in_row : half_krow(wave_u, i) + (lane_v >> 4) < k_left) ? p_off[i] : BUF_OUTSIDE;
        });
    };

    // ---- first tile: its gathered rows are fetched on the spot, the rows of its epilogue go the way of all later ones
    PstTile cur;
    int e_buf = 0; // which of the two epilogue-row buffers holds the current tile's
    auto first_tile = [&]() {
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        cur = entry(0);
        uint32_t q_raw[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            q_raw[i] = need_q_idx ? idx32[2 * ((int64_t)cur.row0 + clamp_row(cur, half_row(wave, i) + (lane >> 3)))] : 0u;
        make_bases(cur);
        static_for<8>([&](auto I) { make_q_off(cur, I, lane, wave, q_raw[I.value]), make_p_off(cur, I, lane, wave); });
        wave_u = wave, lane_v = lane;
        static_for<16>([&](auto P) { issue_piece(0, ordered(P), IC<0>{}); });
        e_buf = 0;
        if (need_e_idx)
            static_for<2>([&](auto M) {
                lds_dma4_raw(idx32 + 2 * ((int64_t)cur.row0 + clamp_row(cur, (wave & 1) * 128 + M.value * 64 + lane)), row_item_lds(PST_ER + M.value, wave));
            });
    };
    walk_len = fill_walk((int)threadIdx.x);
    if (walk_len == 0) return;
    first_tile();

#ifdef XMA_PST_TIMING
    const bool ovl_allowed = !g_pst_no_ovl;
#else
    constexpr bool ovl_allowed = true;
#endif
    [[maybe_unused]] int tile_no = 0;
    for (;; ++tile_no) {
        PST_STAMP(0);
        // Everything derived from the thread index is derived again for every tile behind an opaque copy of it: hoisted
        // out of the tile loop those values would live across the main loop and be spilled.
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        wave_u = wave, lane_v = lane;
        const int wq = (wave & 1) * 128, wp = (wave >> 1) * 128;
        const Bias bias = load_bias(a, cur.e, cur.n0, wp, lane); // behind the first K step: the wait is one for both
        // the first K step and the rows of this tile's epilogue have landed in every wave, the stores of the last
        // epilogue have been handed over and its staging area is dead
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        PST_STAMP(1);

        // One tile ahead: the next tile's schedule entry and rows, and this tile's row scales (their addresses are the
        // epilogue's row indices, fetched a tile ago); all of it lands in LDS during the main loop.  A tile of more than
        // 192 rows with an even number of at least four K steps does this between the MFMAs of its first K step,
        // sets up and loads the first K step of the next tile in its last one
        // (`ovl`); any other tile does it here and behind the loop, with idle matrix pipes.
        const int q_blocks = (cur.rows_valid > wq) ? (cur.rows_valid - wq + 31) >> 5 : 0;
        // uniform over the workgroup: the waves of a tile's lower half (wq == 0) and upper half disagree on q_blocks, so
        // the decision is taken on the tile's row count
        const bool ovl = cur.rows_valid > 128 + 64 && (KT & 1) == 0 && KT >= 4 && ovl_allowed;
        PstTile nxt = {0, 0, 0, 0, 0, 0};
        if (!ovl) {
            nxt = entry(cur.n + 1);
            static_for<ROW_LOADS>([&](auto IT) { prefetch_item(IT, nxt, lane, wave, e_buf); });
        }
        // Two copies of the rest of the tile: the accumulators of the one that overlaps do not have to meet those of the
        // other in the same registers.
        auto rest_of_tile = [&](auto OVL) {
        HalfBase<0> qb;
        HalfBase<WT> pb;
        make_half_base<0>(qb, lds0, wq, lane);
        make_half_base<WT>(pb, lds0 + OP_CHUNKS * 16, wp, lane);
        Half q0, q1, pA, pB;
        static_for<8>([&](auto R) { reader<0, 0, 2>(q0, qb)(R), reader<WT, 0, 2>(pA, pb)(R); });
        PST_STAMP(2);
        // The first half of the second K step's loads goes out between the MFMAs that produce the accumulators, the second
        // half in the first phase of the loop: sixteen in a row would hold up the first MFMAs until the texture unit has
        // taken them all.
        f32x16 acc[4][4];
        init_acc<T>(bias, acc, lane, [&](auto S) {
            constexpr k_schedule::Load l = k_schedule::load_before_loop(S.value);
            if constexpr (l.piece >= 0) issue_piece(l.ahead, IC<l.piece>{}, OVL);
        });
        if constexpr (k_schedule::BARRIER_BEFORE_LOOP)
            XMA_WAIT_READS_AND_BARRIER();
        else
            XMA_WAIT_READS();
        tie_half(q0), tie_half(pA);
        auto main_loop = [&](auto NI_) {
            constexpr int NI = NI_.value, NB0 = NI < 2 ? NI : 2, NB1 = NI > 2 ? 2 : 0;
            // One K step; on entry q0 and p0 hold Q0 and P0 of step kt, on exit q0 and p1 those of step kt + 1.  MODE: what
            // it loads and waits for.
            auto k_step = [&](int kt, Half &p0, Half &p1, auto MODE) {
                constexpr int mode = MODE.value;
                int kt_b = kt + 2;
                asm volatile("" : "+s"(kt_b)); // one address per step, not sixteen running pointers
                [[maybe_unused]] uint32_t nxt_rows[8];
                if constexpr (mode == k_schedule::OVL_LAST) {
                    // the next tile's eight gathered rows, read in one go in front of the step's MFMAs; also when there is
                    // no next tile (nothing is loaded from the addresses then: its buffers are empty)
#pragma unroll
                    for (int i = 0; i < 8; ++i) nxt_rows[i] = row_item(PST_QR, wave, 8 * i + (lane >> 3));
                    make_bases(nxt);
                }
                auto load = [&](auto S, auto PHASE) {
                    constexpr k_schedule::Load l = k_schedule::load_of(mode, PHASE.value, S.value);
                    if constexpr (mode == k_schedule::OVL_LAST) { // addresses in the slots in front of the loads
                        if constexpr (PHASE.value == 0) make_p_off(nxt, S, lane, wave);
                        if constexpr (l.piece >= 0) issue_piece(0, IC<l.piece>{}, IC<1>{});
                        if constexpr (PHASE.value == 1) make_q_off(nxt, S, lane, wave, nxt_rows[S.value]);
                    } else if constexpr (l.piece >= 0) {
                        issue_piece(kt_b - 2 + l.ahead, IC<l.piece>{}, IC<(mode < k_schedule::CHECKED) ? 1 : 0>{});
                    }
                    constexpr int row = k_schedule::row_load_of(mode, PHASE.value, S.value);
                    if constexpr (row >= 0) prefetch_item(IC<row>{}, nxt, lane, wave, e_buf);
                };
                quadrant<T, 0, 0, NB0>(p0, q0, acc, reader<WT, 1, (NI > 0) ? 2 : 0>(p1, pb), [&](auto S) {
                    load(S, IC<0>{});
                });
                XMA_WAIT_READS();
                tie_half(p1);
                quadrant<T, 2, 0, NB0>(p1, q0, acc, reader<0, 1, NB1>(q1, qb), [&](auto S) {
                    load(S, IC<1>{});
                    if constexpr (mode == k_schedule::OVL_FIRST && S.value == 7) nxt = entry(cur.n + 1);
                });
                // {Q0, P0} of step kt + 1 have landed, everybody has read {P1, Q1} of this step
                constexpr int left_b = k_schedule::in_flight_b(mode), left_a = k_schedule::in_flight_a(mode);
                if constexpr (left_b < 0)
                    XMA_WAIT_READS_AND_BARRIER();
                else
                    XMA_WAIT_AND_BARRIER(left_b);
                tie_half(q1);
                flip_half_base(qb), flip_half_base(pb);
                if constexpr (!k_schedule::reads_ahead(mode)) {
                    quadrant<T, 2, 2, NB1>(p1, q1, acc, NoRead(), [&](auto S) { load(S, IC<2>{}); });
                    quadrant<T, 0, 2, NB1>(p0, q1, acc, NoRead(), [&](auto S) { load(S, IC<3>{}); });
                } else {
                    quadrant<T, 2, 2, NB1>(p1, q1, acc, reader<0, 0, NB0>(q0, qb), [&](auto S) { load(S, IC<2>{}); });
                    quadrant<T, 0, 2, NB1>(p0, q1, acc, reader<WT, 0, (NI > 0) ? 2 : 0>(p1, pb), [&](auto S) { load(S, IC<3>{}); });
                    // {P1, Q1} of step kt + 1 have landed, everybody has read {Q0, P0} of it
                    XMA_WAIT_AND_BARRIER(left_a);
                    tie_half(q0), tie_half(p1);
                }
                PST_STEP_STAMP(kt);
            };
            if constexpr (OVL.value != 0) {
                k_step(0, pA, pB, IC<k_schedule::OVL_FIRST>{});
                if (KT == 4) cut_tail();
                k_step(1, pB, pA, IC<k_schedule::OVL_SECOND>{});
                for (int kt = 2; kt < KT - 2; kt += 2) {
                    k_step(kt, pA, pB, IC<k_schedule::STEADY>{});
                    if (kt == KT - 4) cut_tail(); // the next step loads the last one
                    k_step(kt + 1, pB, pA, IC<k_schedule::STEADY>{});
                }
                k_step(KT - 2, pA, pB, IC<k_schedule::OVL_DRAIN>{});
                k_step(KT - 1, pB, pA, IC<k_schedule::OVL_LAST>{});
            } else {
                k_step(0, pA, pB, IC<k_schedule::CHECKED_FIRST>{});
                int kt = 1;
                for (; kt + 1 < KT; kt += 2) {
                    k_step(kt, pB, pA, IC<k_schedule::CHECKED>{});
                    k_step(kt + 1, pA, pB, IC<k_schedule::CHECKED>{});
                }
                if (kt < KT) k_step(kt, pB, pA, IC<k_schedule::CHECKED>{});
            }
        };
        if constexpr (OVL.value != 0) {
            // the waves meet behind their last reads of stage 1; only the next tile's first K step is in flight, into stage 0
            main_loop(IC<4>{});
        } else {
            if (q_blocks > 2)
                main_loop(IC<4>{});
            else if (q_blocks == 2)
                main_loop(IC<2>{});
            else if (q_blocks == 1)
                main_loop(IC<1>{});
            else
                main_loop(IC<0>{});
            XMA_WAIT_LOADS_AND_BARRIER(); // every load has landed, no wave touches the operand tiles any more
        }
        PST_STAMP(3);

        int tid_e = threadIdx.x;
        asm volatile("" : "+v"(tid_e));
        const int lane_e = tid_e & 63, wave_e = __builtin_amdgcn_readfirstlane(tid_e >> 6);
        if constexpr (OVL.value == 0) { // first K step of the next tile: in flight during the epilogue
            wave_u = wave_e, lane_v = lane_e;
            make_bases(nxt);
            static_for<8>([&](auto I) {
                make_q_off(nxt, I, lane_e, wave_e, row_item(PST_QR, wave_e, 8 * I.value + (lane_e >> 3)));
                make_p_off(nxt, I, lane_e, wave_e);
            });
            static_for<16>([&](auto P) { issue_piece(0, ordered(P), IC<0>{}); });
        }
        PST_STAMP(4);
        EpiRows er;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int slot = (i & 1) * 32 + (lane_e & 31);
            const uint32_t s_idx = need_e_idx ? row_item(PST_ER + 2 * e_buf + (i >> 1), wave_e, slot) : 0u;
            er.idx[i] = (int)s_idx;
            er.sc[i] = 1.f;
            if (a.scale) {
                const uint32_t w = row_item(PST_SC + (i >> 1), wave_e, slot);
                er.sc[i] = (s_idx & 1) ? Elem<T>::hi(w) : Elem<T>::lo(w);
            }
        }
        tile_epilogue<T, EPI, 4, 1>(a, acc, smem + PST_STAGING_OFF, cur.row0, cur.rows_valid, cur.n0, tid_e, -1, &er);
        };
        if (ovl)
            rest_of_tile(IC<1>{});
        else
            rest_of_tile(IC<0>{});
        PST_STAMP(5);
#ifdef XMA_PST_TIMING
        if (tile_no == PST_STEP_TILE && threadIdx.x == 0 && blockIdx.x < 256)
            for (int q = 0; q < KT && q < PST_MAX_STEPS; ++q) g_pst_steps[blockIdx.x][q] = ((uint64_t *)(smem + PST_STEP_LDS_OFF))[q];
#endif
        if (!nxt.valid) {
            // the end of the table: usually of the walk; a launch of more than PST_WALK tiles per workgroup refills it and
            // starts over as at the top of the kernel
            XMA_WAIT_LOADS_AND_BARRIER(); // (no load into LDS is in flight when the workgroup ends)
            if ((int64_t)blockIdx.x + (int64_t)walk_pos * gridDim.x >= a.grid_main) break;
            walk_len = fill_walk((int)threadIdx.x);
            if (walk_len == 0) break;
            first_tile();
            continue;
        }
        cur = nxt;
        e_buf ^= 1;
    }
}

// ------------------------------------------------------------------------------------------------
// dW kernel: DW[e][o][i] = sum_n DY[n][o] X[n][i]; both operands are token-major = transposed sources; the K loop
// runs over the expert's row range, k-rows past its end come from the zero page.
//   GQ / GP = 1: the rows of dY / X are taken through sorted_scattered_idxs (index / fan_out); 0: grouped order
// ------------------------------------------------------------------------------------------------
constexpr int DW_BAND = 4;
#ifdef XMA_PST_TIMING
// timing build: shader clock counter of the first DW_TIMING_TILES workgroups at the start of the kernel, in front of and
// behind the K loop and at the end, and the tile's K step count
constexpr int DW_TIMING_TILES = 8192;
__device__ uint64_t g_dw_cycles[DW_TIMING_TILES][6];
#define DW_STAMP(k)                                                                   \
    do {                                                                              \
        if (threadIdx.x == 0 && blockIdx.x < DW_TIMING_TILES)                          \
            g_dw_cycles[blockIdx.x][k] = (k) == 4 ? (uint64_t)KT : __builtin_amdgcn_s_memtime(); \
    } while (0)
#else
#define DW_STAMP(k) \
    do {            \
    } while (0)
#endif
template <typename T, int GQ, int GP>
__global__ __launch_bounds__(GEMM_THREADS, 1) void grouped_gemm_dw_kernel(const DwArgs a) {
    constexpr int GATHER = GQ | GP;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    u32x4 *tiles = (u32x4 *)smem;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int OT = (a.N_out + 255) / 256, IT = (a.K_in + 255) / 256;
    // Tile walk: inside an expert the tiles are taken in bands of DW_BAND tile rows, down the band first, so that the 32
    // consecutive tiles an XCD gets from xcd_remap form a DW_BAND x (32 / DW_BAND) block that shares DW_BAND dY panels and
    // 32 / DW_BAND X panels in that XCD's L2 (a row-by-row walk shares 1 + 32).
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    const int rem = L % (OT * IT);
    // Experts are taken in the order of decreasing row count (equal counts: lower index first), the longest K loops
    // first: a tile's duration is proportional to its expert's rows, and with skewed routing a large expert that came up
    // last would keep a few compute units busy long after all others have finished.  Every wave ranks the experts in
    // registers (lane = expert); with more experts than lanes the order stays the index order.
    int e = L / (OT * IT);
    if (a.E <= WAVE) {
        const int64_t hi = a.offs[lane < a.E ? lane : a.E - 1];
        int64_t lo = __shfl_up(hi, 1);
        if (lane == 0) lo = 0;
        const int cnt = (lane < a.E) ? (int)(hi - lo) : -1;
        int rank = 0;
        for (int i = 0; i < a.E; ++i) {
            const int ci = __builtin_amdgcn_readlane(cnt, i);
            rank += (ci > cnt || (ci == cnt && i < lane)) ? 1 : 0;
        }
        e = __builtin_ctzll(__ballot(rank == e && lane < a.E)); // exactly one lane
    }
    const int band = rem / (DW_BAND * IT), in_band = rem % (DW_BAND * IT);
    const int band_rows = (OT - band * DW_BAND < DW_BAND) ? OT - band * DW_BAND : DW_BAND;
    const int o0 = (band * DW_BAND + in_band % band_rows) * 256, i0 = (in_band / band_rows) * 256;
    const int64_t row_lo = e ? a.offs[e - 1] : 0, row_hi = a.offs[e];
    const int rows = (int)(row_hi - row_lo);
    const int KT = (rows + BK - 1) / BK;
    DW_STAMP(0);
    DW_STAMP(4);
    const uint16_t *zero = (const uint16_t *)g_zero_page;
    const int q_max_chunk = ((a.N_out - o0) >> 3) - 1, p_max_chunk = ((a.K_in - i0) >> 3) - 1;
    const int kr_lane = wave * 16 + (lane >> 5); // this lane's k-rows of a step: kr_lane + 2 j, j = 0..7

    // Per-lane column offsets (elements) of the 8 pieces of each operand; rows change every step.  For an operand in
    // grouped order the row is row_lo + 64 kt + kr, so the piece pointer advances by a uniform 64 ld per step.
    int q_col[8], p_col[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        int cq = transposed_lane_chunk(j, lane), cp = cq;
        if (cq > q_max_chunk) cq = q_max_chunk; // columns past the edge are masked at the store
        if (cp > p_max_chunk) cp = p_max_chunk;
        q_col[j] = o0 + cq * 8;
        p_col[j] = i0 + cp * 8;
    }
    // Per-lane byte pointers of the 8 pieces of each operand: for an operand in grouped order the address of step 0
    // (the row is row_lo + 64 kt + kr, so a step adds a uniform 64 rows); for a gathered operand the column position in
    // row 0, to which token * row pitch is added (one 32 x 32 -> 64-bit multiply-add per piece).
    const uint32_t lddy_b = (uint32_t)a.lddy * 2, ldx_b = (uint32_t)a.ldx * 2;
    const char *q_base[8], *p_base[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        q_base[j] = (const char *)(a.DY + q_col[j]) + (GQ ? 0 : (row_lo + kr_lane + 2 * j) * (int64_t)lddy_b);
        p_base[j] = (const char *)(a.X + p_col[j]) + (GP ? 0 : (row_lo + kr_lane + 2 * j) * (int64_t)ldx_b);
    }

    // Scattered indices of this lane's 8 tokens of the step that is loaded next.  They are fetched one step ahead with
    // inline assembly (low dword of the int64 index): the compiler would guard the later use of a loop-carried loaded
    // register with a wait of its own choosing; here the wait is the vmcnt(0) in front of each step's barrier, and
    // use_idx() ties the registers to a point behind it.  FULL: all rows of the step lie inside the expert, the address
    // is one per-lane pointer plus an immediate.
    uint32_t idx_next[8];
    const int64_t *idx_lane = a.idx + row_lo + kr_lane;
    auto load_idx_one = [&](int kt, auto J, auto FULL) {
        constexpr int j = J.value;
        if constexpr (FULL.value) {
            const int64_t *src = idx_lane + (int64_t)kt * BK;
            asm volatile("global_load_dword %0, %1, off offset:%2" : "=v"(idx_next[j]) : "v"(src), "n"(16 * j) : "memory");
        } else {
            int r = kt * BK + kr_lane + 2 * j;
            if (r >= rows) r = rows - 1; // clamped, never predicated
            const int64_t *src = a.idx + row_lo + r;
            asm volatile("global_load_dword %0, %1, off" : "=v"(idx_next[j]) : "v"(src) : "memory");
        }
    };
    auto load_idx = [&](int kt) { static_for<8>([&](auto J) { load_idx_one(kt, J, IC<0>{}); }); };
    auto use_idx = [&]() {
        asm volatile("s_waitcnt vmcnt(0)"
                     : "+v"(idx_next[0]), "+v"(idx_next[1]), "+v"(idx_next[2]), "+v"(idx_next[3]), "+v"(idx_next[4]),
                       "+v"(idx_next[5]), "+v"(idx_next[6]), "+v"(idx_next[7]));
    };
    // piece 0..15 of K step kt (0..7 = dY tile, 8..15 = X tile); FULL: step kt exists and lies inside the expert's rows
    auto issue_piece = [&](int kt, auto PIECE, auto FULL) {
        constexpr int piece = PIECE.value, j = piece & 7;
        if constexpr (!FULL.value) {
            if (kt >= KT) return; // uniform
        }
        u32x4 *dst = tiles + (kt & 1) * STAGE_CHUNKS + (piece >> 3) * OP_CHUNKS + j * 64 + wave * 512;
        const char *src;
        if constexpr (piece < 8) {
            if (GQ)
                src = q_base[j] + (uint64_t)fastdiv(idx_next[j], a.dy_div) * lddy_b;
            else
                src = q_base[j] + (uint64_t)(uint32_t)(kt * BK) * lddy_b;
        } else {
            if (GP)
                src = p_base[j] + (uint64_t)fastdiv(idx_next[j], a.x_div) * ldx_b;
            else
                src = p_base[j] + (uint64_t)(uint32_t)(kt * BK) * ldx_b;
        }
        if constexpr (!FULL.value) {
            if (kt == KT - 1) { // uniform branch: k-rows past the expert's range come from the zero page
                asm volatile("" ::: "memory"); // keeps this rare path a branch
                if (kt * BK + kr_lane + 2 * j >= rows) src = (const char *)zero;
            }
        }
        lds_dma16((const uint16_t *)src, dst);
    };

    f32x16 acc[4][4];
    zero_acc(acc);
    const int wq = (wave & 1) * 128, wp = (wave >> 1) * 128;
    if (KT > 0) {
        // VMEM order per wave: idx(0) | dma(0) idx(1) | dma(1)[0..7] idx(2)? - see below; in the loop the indices of a
        // step are always loaded before a vmcnt(0) that precedes their use.
        const uint32_t lds0 = lds_addr_of(smem);
        FragBase<1> qb, pb;
        make_frag_base<1>(qb, lds0, wq, lane);
        make_frag_base<1>(pb, lds0 + OP_CHUNKS * 16, wp, lane);
        // the operand that is not gathered needs no index: its first step goes out while the indices are on their way
        if (GATHER) load_idx(0);
        if (!GQ) static_for<8>([&](auto P) { issue_piece(0, P, IC<0>{}); });
        if (!GP) static_for<8>([&](auto P) { issue_piece(0, IC<8 + P.value>{}, IC<0>{}); });
        if (GATHER) use_idx();
        if (GQ) static_for<8>([&](auto P) { issue_piece(0, P, IC<0>{}); });
        if (GP) static_for<8>([&](auto P) { issue_piece(0, IC<8 + P.value>{}, IC<0>{}); });
        __builtin_amdgcn_sched_barrier(0);
        if (GATHER) {
            load_idx(1);
            use_idx(); // vmcnt(0): step 0 has landed as well
        }
        static_for<8>([&](auto P) { issue_piece(1, P, IC<0>{}); });
        __builtin_amdgcn_sched_barrier(0);
        // step 0 has landed in every wave; behind it at most the first half of step 1 (none if this is the only step)
        if (KT > 1)
            asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        Frags f0, f1;
        load_frags<1, 1, 0>(f0, pb, qb);
        DW_STAMP(1);
        // one K step; FULL: steps kt + 1 and kt + 2 lie completely inside the expert's rows
        auto k_step = [&](int kt, auto FULL) {
            // idx_next holds the indices of step kt + 1 here; the second half of that step's loads goes out now, then
            // the indices of step kt + 2 are requested (they land before the barrier's vmcnt(0))
            mma_step<T, 1, 1, 1>(f0, f1, pb, qb, acc, [&](auto G) { issue_piece(kt + 1, IC<8 + G.value>{}, FULL); });
            mma_step<T, 1, 1, 2>(f1, f0, pb, qb, acc, [&](auto G) {
                if constexpr (GATHER != 0) load_idx_one(kt + 2, G, FULL);
            });
            mma_step<T, 1, 1, 3>(f0, f1, pb, qb, acc, NoHook());
            XMA_WAIT_LOADS_AND_BARRIER();
            if (GATHER) use_idx();
            flip_stage(pb);
            flip_stage(qb);
            mma_step<T, 1, 1, 0>(f1, f0, pb, qb, acc, [&](auto G) { issue_piece(kt + 2, G, FULL); });
        };
        const int KT_full = rows / BK;
        int kt = 0;
        for (; kt + 2 < KT_full; ++kt) k_step(kt, IC<1>{});
        for (; kt < KT; ++kt) k_step(kt, IC<0>{});
        wait_frags(f0); // read ahead and not used: see the forward kernel
        XMA_WAIT_ALL_LOADS();
        DW_STAMP(2);
    }

    // lane owns DW row o (from the Q tile), 4 consecutive in-features per quad; each 32-row block is staged in a
    // wave-private LDS area and leaves as whole rows (see the forward kernel's epilogue)
    XMA_WAIT_LOADS_AND_BARRIER(); // no wave reads the operand tiles any more
    const int lrow = lane & 31, lhalf = lane >> 5;
    uint16_t *DWe = a.DW + (int64_t)e * a.dw_es;
    unsigned char *stage = smem + wave * EPI_WAVE_BYTES;
    unsigned char *z_w = stage + lrow * EPI_Z_STRIDE + lhalf * 8;
    const unsigned char *z_r = stage + (lane >> 4) * EPI_Z_STRIDE + (lane & 15) * 16;
    const int cz = i0 + wp + (lane & 15) * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int obase = o0 + wq + i * 32;
        if (obase >= a.N_out) break; // wave-uniform
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32x2 v = {Elem<T>::pack(acc[j][i][4 * g], acc[j][i][4 * g + 1]),
                           Elem<T>::pack(acc[j][i][4 * g + 2], acc[j][i][4 * g + 3])};
                *(u32x2 *)(z_w + (j * 32 + g * 8) * 2) = v;
            }
        wave_lds_sync();
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int o = obase + 4 * it + (lane >> 4);
            const u32x4 v = *(const u32x4 *)(z_r + it * 4 * EPI_Z_STRIDE);
            if (o < a.N_out && cz < a.K_in) *(u32x4 *)(DWe + (int64_t)o * a.lddw + cz) = v;
        }
        wave_lds_sync(); // the next block overwrites the area
    }
    DW_STAMP(3);
}

inline int device_cus();
template <typename T, int WT, int EPI> int launch_fwd(const FwdArgs &a, hipStream_t st) {
    int rc;
    const int cus = device_cus();
    // The persistent kernel fetches a row scale as the aligned dword around it and addresses the operands of a tile with
    // 32-bit byte offsets from a uniform base: 256 rows of W or of a grouped X, any row of a gathered X, any row scale (the
    // dword of the last one has to end within the 2^32 - 16 bytes of a buffer, or it reads zeros).
    const int64_t x_rows = a.x_grouped ? 256 : (a.M + a.fan_out - 1) / a.fan_out;
    const bool offsets_fit = x_rows * a.ldx * 2 < ((int64_t)1 << 32) && (int64_t)256 * a.ldw * 2 < ((int64_t)1 << 32) &&
                             (!a.scale || 2 * a.M <= (int64_t)0xfffffff0);
    // The persistent kernel exists for the operand layouts the layer launches: x @ W^T with any epilogue, dy @ W with a
    // plain store or the SwiGLU backward.  (dy @ W with the SwiGLU forward epilogue is reachable through the C ABI only: not
    // worth another 120 KB of code per type.)
    constexpr bool persistent_variant = !(WT == 1 && EPI == XMA_ROCM_EPI_SWIGLU);
    bool persistent = false;
    if constexpr (persistent_variant) {
        if (a.E <= PST_MAX_E && cus > 0 && ((uintptr_t)a.scale & 3) == 0 && offsets_fit && row_offsets_fit(a)) {
            // whole tiles: one persistent workgroup per compute unit
            if ((rc = gemm_set_smem(grouped_gemm_persistent_kernel<T, WT, EPI>, PST_SMEM_BYTES))) return rc;
            const int launch_grid = cus < a.grid_main ? cus : a.grid_main;
            grouped_gemm_persistent_kernel<T, WT, EPI><<<launch_grid, GEMM_THREADS, PST_SMEM_BYTES, st>>>(a);
            if ((rc = xma_check_launch("grouped_gemm_persistent_kernel"))) return rc;
            persistent = true;
        }
    }
    if (!persistent) {
        if ((rc = gemm_set_smem(grouped_gemm_kernel<T, WT, EPI, ROLE_TILES>, GEMM_SMEM_BYTES))) return rc;
        int launch_grid = a.grid_main;
        if (fwd_persistent(EPI, ROLE_TILES) && cus > 0 && cus < launch_grid) launch_grid = cus;
        grouped_gemm_kernel<T, WT, EPI, ROLE_TILES><<<launch_grid, GEMM_THREADS, GEMM_SMEM_BYTES, st>>>(a);
        if ((rc = xma_check_launch("grouped_gemm_kernel"))) return rc;
    }
    if (!a.partial) return XMA_ROCM_OK;
    // the tiles of the last round as K slices (no epilogue: one instantiation serves all), then their sum + epilogue
    if ((rc = gemm_set_smem(grouped_gemm_kernel<T, WT, XMA_ROCM_EPI_STORE, ROLE_SLICES>, GEMM_SMEM_BYTES))) return rc;
    grouped_gemm_kernel<T, WT, XMA_ROCM_EPI_STORE, ROLE_SLICES><<<a.split_cus, GEMM_THREADS, GEMM_SMEM_BYTES, st>>>(a);
    if ((rc = xma_check_launch("grouped_gemm_kernel (K slices)"))) return rc;
    if ((rc = gemm_set_smem(grouped_gemm_fixup_kernel<T, EPI>, GEMM_SMEM_BYTES))) return rc;
    grouped_gemm_fixup_kernel<T, EPI><<<4 * a.split_cus, GEMM_THREADS, GEMM_SMEM_BYTES, st>>>(a);
    return xma_check_launch("grouped_gemm_fixup_kernel");
}

template <typename T, int GQ, int GP> int launch_dw(const DwArgs &a, int grid, hipStream_t st) {
    int rc = gemm_set_smem(grouped_gemm_dw_kernel<T, GQ, GP>, GEMM_SMEM_BYTES);
    if (rc) return rc;
    grouped_gemm_dw_kernel<T, GQ, GP><<<grid, GEMM_THREADS, GEMM_SMEM_BYTES, st>>>(a);
    return xma_check_launch("grouped_gemm_dw_kernel");
}

template <typename T> int dispatch_dw(const DwArgs &a, int grid, hipStream_t st) {
    if (a.dy_grouped) return a.x_grouped ? launch_dw<T, 0, 0>(a, grid, st) : launch_dw<T, 0, 1>(a, grid, st);
    return a.x_grouped ? launch_dw<T, 1, 0>(a, grid, st) : launch_dw<T, 1, 1>(a, grid, st);
}

template <typename T> int dispatch_fwd(const FwdArgs &a, int wt, int epi, hipStream_t st) {
    if (wt == 0) {
        if (epi == XMA_ROCM_EPI_STORE) return launch_fwd<T, 0, XMA_ROCM_EPI_STORE>(a, st);
        if (epi == XMA_ROCM_EPI_SWIGLU) return launch_fwd<T, 0, XMA_ROCM_EPI_SWIGLU>(a, st);
        return launch_fwd<T, 0, XMA_ROCM_EPI_SWIGLU_BWD>(a, st);
    }
    if (epi == XMA_ROCM_EPI_STORE) return launch_fwd<T, 1, XMA_ROCM_EPI_STORE>(a, st);
    if (epi == XMA_ROCM_EPI_SWIGLU) return launch_fwd<T, 1, XMA_ROCM_EPI_SWIGLU>(a, st);
    if (a.dots) return a.aux2 ? launch_fwd<T, 1, EPI_SWIGLU_BWD_SCALED_ACT_DOTS>(a, st) : launch_fwd<T, 1, EPI_SWIGLU_BWD_DOTS>(a, st);
    if (a.aux2) return launch_fwd<T, 1, EPI_SWIGLU_BWD_SCALED_ACT>(a, st);
    return launch_fwd<T, 1, XMA_ROCM_EPI_SWIGLU_BWD>(a, st);
}

// Compute units of the current device (tiles that run at the same time), looked up once per device.
inline int device_cus() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
        cached[dev].store(n, std::memory_order_relaxed); // every thread that races here stores the same value
    }
    return n;
}

// Launches of fewer rounds than this may split the tiles of their last round over the idle CUs.
constexpr int64_t SPLIT_MAX_ROUNDS = 12;

inline size_t fwd_workspace_bytes(int64_t M, int32_t N, int32_t K, int32_t E) {
    const int cus = device_cus();
    if (cus <= 0) return 0;
    // a tile is cut into at least two slices of SPLIT_MIN_STEPS K steps or not at all: short K never splits, and the two
    // launches that would find nothing to do are not made
    if ((K + BK - 1) / BK < 2 * SPLIT_MIN_STEPS) return 0;
    const int64_t tiles = (M / BM + E) * ((N + BN - 1) / BN);
    if (tiles > SPLIT_MAX_ROUNDS * cus) return 0;
    return (size_t)cus * BM * BN * sizeof(float);
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

} // namespace xma_rocm

using namespace xma_rocm;

#ifdef XMA_GROUPED_GEMM_F16 // the kernels for fp16 are a translation unit of their own (grouped_gemm_f16.hip), without the entry points
int grouped_fwd_f16(const FwdArgs &a, int wt, int epi, hipStream_t st) { return dispatch_fwd<_Float16>(a, wt, epi, st); }
int grouped_dw_f16(const DwArgs &a, int grid, hipStream_t st) { return dispatch_dw<_Float16>(a, grid, st); }
#else

static int scatter2scatter_impl(const void *X, int64_t ldx, const void *W, int64_t w_expert_stride, int64_t ldw,
                                int w_is_kn, const int64_t *sorted_scattered_idxs, const int64_t *expert_offsets,
                                void *out, int64_t ldo, void *aux, int64_t ldaux, void *aux2, int64_t ldaux2,
                                const void *row_scale, const void *bias, int64_t bias_expert_stride, int64_t M, int32_t N,
                                int32_t K, int32_t E, int32_t fan_out, int x_grouped, int y_grouped, int epilogue, int dtype,
                                void *workspace, size_t workspace_bytes, void *stream, float *dots = nullptr) {
    XMA_REQUIRE(dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16 || dtype == XMA_ROCM_F32, XMA_ROCM_EUNSUPPORTED,
                "scatter2scatter: dtype %d", dtype);
    XMA_REQUIRE(epilogue >= XMA_ROCM_EPI_STORE && epilogue <= XMA_ROCM_EPI_SWIGLU_BWD, XMA_ROCM_EINVAL,
                "scatter2scatter: epilogue %d", epilogue);
    XMA_REQUIRE(M >= 0 && M < ((int64_t)1 << 31) && N >= 8 && K >= 8 && E >= 1 && fan_out >= 1, XMA_ROCM_EINVAL,
                "scatter2scatter: M=%lld N=%d K=%d E=%d fan_out=%d", (long long)M, N, K, E, fan_out);
    XMA_REQUIRE(N % 8 == 0 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldo % 8 == 0 && w_expert_stride % 8 == 0,
                XMA_ROCM_EUNSUPPORTED, "scatter2scatter: N=%d K=%d ldx=%lld ldw=%lld ldo=%lld must be multiples of 8", N,
                K, (long long)ldx, (long long)ldw, (long long)ldo);
    XMA_REQUIRE(E <= 16384, XMA_ROCM_EUNSUPPORTED, "scatter2scatter: E=%d > 16384", E);
    if (M == 0) return XMA_ROCM_OK;
    XMA_REQUIRE(X && W && expert_offsets && aligned16(X) && aligned16(W), XMA_ROCM_EINVAL,
                "scatter2scatter: null or misaligned operand");
    XMA_REQUIRE(sorted_scattered_idxs || (x_grouped && y_grouped && !row_scale), XMA_ROCM_EINVAL,
                "scatter2scatter: sorted_scattered_idxs is required unless everything is grouped");
    if (epilogue == XMA_ROCM_EPI_STORE) {
        XMA_REQUIRE(out && aligned16(out), XMA_ROCM_EINVAL, "scatter2scatter: out is null or misaligned");
    } else if (epilogue == XMA_ROCM_EPI_SWIGLU) {
        XMA_REQUIRE(aux && aligned16(aux) && ldaux % 8 == 0 && N % 16 == 0, XMA_ROCM_EINVAL,
                    "scatter2scatter: SWIGLU needs aux (M, N/2), ldaux %% 8 == 0, N %% 16 == 0");
        XMA_REQUIRE(!out || aligned16(out), XMA_ROCM_EINVAL, "scatter2scatter: misaligned out");
    } else {
        XMA_REQUIRE(out && aux && aligned16(out) && aligned16(aux) && ldaux % 8 == 0 && y_grouped, XMA_ROCM_EINVAL,
                    "scatter2scatter: SWIGLU_BWD needs out, aux (z) and y_grouped");
    }
    XMA_REQUIRE(!aux2 || (epilogue == XMA_ROCM_EPI_SWIGLU_BWD && aligned16(aux2) && ldaux2 % 8 == 0 && ldaux2 >= N),
                XMA_ROCM_EINVAL, "scatter2scatter: scaled activations go with SWIGLU_BWD, 16-byte aligned rows");
    XMA_REQUIRE(!aux2 || (dtype != XMA_ROCM_F32 && w_is_kn), XMA_ROCM_EUNSUPPORTED,
                "scatter2scatter: scaled activations need bf16 / fp16 and W[e] as (K, N) with N contiguous (dy @ W)");
    XMA_REQUIRE(!bias || (aligned16(bias) && bias_expert_stride % 8 == 0 && bias_expert_stride >= 0 &&
                          epilogue != XMA_ROCM_EPI_SWIGLU_BWD),
                XMA_ROCM_EINVAL, "scatter2scatter: bias (E, N) must be 16-byte aligned with an expert stride that is a "
                                 "multiple of 8 elements, and goes with the STORE and SWIGLU epilogues");
    FwdArgs a;
    a.bias = (const uint16_t *)bias;
    a.bias_es = bias_expert_stride;
    a.X = (const uint16_t *)X;
    a.ldx = ldx;
    a.W = (const uint16_t *)W;
    a.w_es = w_expert_stride;
    a.ldw = ldw;
    a.idx = sorted_scattered_idxs;
    a.offs = expert_offsets;
    a.out = (uint16_t *)out;
    a.ldo = ldo;
    a.aux = (uint16_t *)aux;
    a.ldaux = ldaux;
    a.aux2 = (uint16_t *)aux2;
    a.ldaux2 = ldaux2;
    a.scale = (const uint16_t *)row_scale;
    a.M = M;
    a.N = N;
    a.K = K;
    a.E = E;
    a.fan_out = fan_out;
    a.fan_div = make_fastdiv((uint32_t)(x_grouped ? 1 : fan_out));
    a.x_grouped = x_grouped;
    a.y_grouped = y_grouped;
    a.partial = nullptr;
    a.split_cus = 0;
    a.grid_main = 0;
    a.erf_form = 0;
    a.dots = dots;
    a.dots_ld = (uint32_t)((N + 127) / 128);
    a.dots_bytes = dots ? (uint32_t)(M * a.dots_ld * 4) : 0u;
    if (dtype == XMA_ROCM_F32) return f32_scatter2scatter(a, w_is_kn ? 1 : 0, epilogue, (hipStream_t)stream);
    const int64_t NT = (N + BN - 1) / BN;
    const int64_t max_m_tiles = M / BM + E; // sum_e ceil(c_e / BM) <= floor(M / BM) + E
    const int64_t grid = max_m_tiles * NT;
    XMA_REQUIRE(grid < ((int64_t)1 << 30), XMA_ROCM_EUNSUPPORTED, "scatter2scatter: grid too large");
    a.grid_main = (int)grid;
    a.partial = nullptr;
    a.split_cus = 0;
    const size_t ws_need = fwd_workspace_bytes(M, N, K, E);
    if (workspace && ws_need) {
        XMA_REQUIRE(workspace_bytes >= ws_need && aligned16(workspace), XMA_ROCM_EWORKSPACE,
                    "scatter2scatter: workspace of %zu bytes, %zu needed (16-byte aligned)", workspace_bytes, ws_need);
        a.partial = (float *)workspace;
        a.split_cus = device_cus();
    }
    hipStream_t st = (hipStream_t)stream;
    if (dtype == XMA_ROCM_BF16) return dispatch_fwd<__bf16>(a, w_is_kn ? 1 : 0, epilogue, st);
    return grouped_fwd_f16(a, w_is_kn ? 1 : 0, epilogue, st);
}

extern "C" int xma_rocm_scatter2scatter(const void *X, int64_t ldx, const void *W, int64_t w_expert_stride, int64_t ldw,
                                        int w_is_kn, const int64_t *sorted_scattered_idxs,
                                        const int64_t *expert_offsets, void *out, int64_t ldo, void *aux, int64_t ldaux,
                                        const void *row_scale, int64_t M, int32_t N, int32_t K, int32_t E,
                                        int32_t fan_out, int x_grouped, int y_grouped, int epilogue, int dtype,
                                        void *workspace, size_t workspace_bytes, void *stream) {
    return scatter2scatter_impl(X, ldx, W, w_expert_stride, ldw, w_is_kn, sorted_scattered_idxs, expert_offsets, out, ldo,
                                aux, ldaux, nullptr, 0, row_scale, nullptr, 0, M, N, K, E, fan_out, x_grouped, y_grouped,
                                epilogue, dtype, workspace, workspace_bytes, stream);
}

extern "C" int xma_rocm_scatter2scatter_bias(const void *X, int64_t ldx, const void *W, int64_t w_expert_stride,
                                             int64_t ldw, int w_is_kn, const int64_t *sorted_scattered_idxs,
                                             const int64_t *expert_offsets, void *out, int64_t ldo, void *aux,
                                             int64_t ldaux, const void *row_scale, const void *bias,
                                             int64_t bias_expert_stride, int64_t M, int32_t N, int32_t K, int32_t E,
                                             int32_t fan_out, int x_grouped, int y_grouped, int epilogue, int dtype,
                                             void *workspace, size_t workspace_bytes, void *stream) {
    return scatter2scatter_impl(X, ldx, W, w_expert_stride, ldw, w_is_kn, sorted_scattered_idxs, expert_offsets, out, ldo,
                                aux, ldaux, nullptr, 0, row_scale, bias, bias_expert_stride, M, N, K, E, fan_out, x_grouped,
                                y_grouped, epilogue, dtype, workspace, workspace_bytes, stream);
}

extern "C" int xma_rocm_down_projection_dx_swiglu(const void *dY, int64_t lddy, const void *W, int64_t w_expert_stride,
                                                  int64_t ldw, const int64_t *sorted_scattered_idxs,
                                                  const int64_t *expert_offsets, const void *z, int64_t ldz, void *dz,
                                                  int64_t lddz, void *scaled_act, int64_t ld_scaled_act,
                                                  const void *row_scale, int64_t M, int32_t N, int32_t K, int32_t E,
                                                  int32_t fan_out, int dtype, void *workspace, size_t workspace_bytes,
                                                  void *stream) {
    XMA_REQUIRE(dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16, XMA_ROCM_EUNSUPPORTED,
                "down_projection_dx_swiglu: dtype %d (bf16 and fp16 only)", dtype);
    XMA_REQUIRE(row_scale && scaled_act, XMA_ROCM_EINVAL, "down_projection_dx_swiglu: row_scale and scaled_act are required");
    return scatter2scatter_impl(dY, lddy, W, w_expert_stride, ldw, 1, sorted_scattered_idxs, expert_offsets, dz, lddz,
                                const_cast<void *>(z), ldz, scaled_act, ld_scaled_act, row_scale, nullptr, 0, M, N, K, E,
                                fan_out, 0, 1, XMA_ROCM_EPI_SWIGLU_BWD, dtype, workspace, workspace_bytes, stream);
}

int xma_down_projection_dx_dots(const void *dY, int64_t lddy, const void *W, int64_t w_expert_stride, int64_t ldw,
                                const int64_t *sorted_scattered_idxs, const int64_t *expert_offsets, const void *z, int64_t ldz, void *dz,
                                int64_t lddz, void *scaled_act, int64_t ld_scaled_act, const void *row_scale, int64_t M, int32_t N,
                                int32_t K, int32_t E, int32_t fan_out, int dtype, void *workspace, size_t workspace_bytes, void *stream,
                                float *dots) {
    XMA_REQUIRE(M * ((N + 127) / 128) < ROUTER_GRADIENT_MAX, XMA_ROCM_EUNSUPPORTED, "down_projection_dx_dots: M=%lld N=%d (M ceil(N / 128) < 2^30 - 4)", (long long)M, N);
    XMA_REQUIRE(row_scale && dots && (dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16), XMA_ROCM_EINVAL, "down_projection_dx_dots: dtype %d, row_scale and dots are required", dtype);
    return scatter2scatter_impl(dY, lddy, W, w_expert_stride, ldw, 1, sorted_scattered_idxs, expert_offsets, dz, lddz,
                                const_cast<void *>(z), ldz, scaled_act, ld_scaled_act, row_scale, nullptr, 0, M, N, K, E,
                                fan_out, 0, 1, XMA_ROCM_EPI_SWIGLU_BWD, dtype, workspace, workspace_bytes, stream, dots);
}

// the K slices of the launch, then the products of rows and 128 columns
extern "C" size_t xma_rocm_down_projection_dx_swiglu_router_workspace_bytes(int64_t M, int32_t N, int32_t K, int32_t E) {
    if (M <= 0 || N <= 0 || K <= 0 || E <= 0) return 0;
    return (fwd_workspace_bytes(M, N, K, E) + 255) / 256 * 256 + (size_t)M * ((N + 127) / 128) * sizeof(float);
}

extern "C" int xma_rocm_down_projection_dx_swiglu_router(const void *dY, int64_t lddy, const void *W, int64_t w_expert_stride,
                                                         int64_t ldw, const int64_t *sorted_scattered_idxs,
                                                         const int64_t *expert_offsets, const void *z, int64_t ldz, void *dz,
                                                         int64_t lddz, void *scaled_act, int64_t ld_scaled_act,
                                                         const void *row_scale, void *d_row_scale, int64_t M, int32_t N, int32_t K,
                                                         int32_t E, int32_t fan_out, int dtype, void *workspace,
                                                         size_t workspace_bytes, void *stream) {
    XMA_REQUIRE(fan_out >= 1 && fan_out <= 32 && M >= 0 && M % fan_out == 0 && (M == 0 || d_row_scale), XMA_ROCM_EINVAL,
                "down_projection_dx_swiglu_router: fan_out=%d M=%lld (at most 32, M a multiple), d_row_scale is required", fan_out, (long long)M);
    const size_t need = xma_rocm_down_projection_dx_swiglu_router_workspace_bytes(M, N, K, E);
    XMA_REQUIRE(M == 0 || (workspace && aligned16(workspace) && workspace_bytes >= need), XMA_ROCM_EWORKSPACE,
                "down_projection_dx_swiglu_router: workspace of %zu bytes, %zu needed (16-byte aligned)", workspace_bytes, need);
    if (M == 0) return XMA_ROCM_OK;
    const int64_t parts = (N + 127) / 128;
    float *dots = (float *)((char *)workspace + need) - M * parts;
    const int rc = xma_down_projection_dx_dots(dY, lddy, W, w_expert_stride, ldw, sorted_scattered_idxs, expert_offsets, z, ldz, dz, lddz,
                                               scaled_act, ld_scaled_act, row_scale, M, N, K, E, fan_out, dtype, workspace,
                                               workspace_bytes, stream, dots);
    if (rc) return rc;
    return xma_dots_router_bwd(dots, parts, nullptr, nullptr, M / fan_out, E, fan_out, dtype, d_row_scale, (hipStream_t)stream);
}

#ifdef XMA_PST_TIMING
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_times(void *host_out) {
    return (int)hipMemcpyFromSymbol(host_out, HIP_SYMBOL(g_pst_times), sizeof(g_pst_times));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_cycles(void *host_out) {
    return (int)hipMemcpyFromSymbol(host_out, HIP_SYMBOL(g_pst_cycles), sizeof(g_pst_cycles));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_steps(void *host_out) {
    return (int)hipMemcpyFromSymbol(host_out, HIP_SYMBOL(g_pst_steps), sizeof(g_pst_steps));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_dw_cycles(void *host_out) {
    return (int)hipMemcpyFromSymbol(host_out, HIP_SYMBOL(g_dw_cycles), sizeof(g_dw_cycles));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_band(int v) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_pst_band), &v, sizeof(v));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_no_ovl(int v) {
    return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_pst_no_ovl), &v, sizeof(v));
}
extern "C" __attribute__((visibility("default"))) int xma_rocm_debug_pst_reset(void) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_pst_times)) != hipSuccess) return -1;
    return (int)hipMemset(p, 0, sizeof(g_pst_times));
}
#endif

extern "C" size_t xma_rocm_scatter2scatter_workspace_bytes(int64_t M, int32_t N, int32_t K, int32_t E) {
    if (M <= 0 || N <= 0 || K <= 0 || E <= 0) return 0;
    return fwd_workspace_bytes(M, N, K, E);
}

int xma_group_bwd_W(const void *DY, int64_t lddy, int dy_grouped, int32_t dy_fan_out, const void *dy_scale, const void *X, int64_t ldx, int x_grouped,
                    int32_t x_fan_out, const int64_t *sorted_scattered_idxs, const int64_t *expert_offsets, void *DW, int64_t dw_expert_stride,
                    int64_t lddw, int32_t N_out, int32_t K_in, int32_t E, int64_t M, int dtype, void *stream) {
    XMA_REQUIRE(dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16 || dtype == XMA_ROCM_F32, XMA_ROCM_EUNSUPPORTED,
                "group_bwd_W: dtype %d", dtype);
    XMA_REQUIRE(N_out >= 8 && K_in >= 8 && E >= 1 && dy_fan_out >= 1 && x_fan_out >= 1, XMA_ROCM_EINVAL,
                "group_bwd_W: N_out=%d K_in=%d E=%d", N_out, K_in, E);
    XMA_REQUIRE(N_out % 8 == 0 && K_in % 8 == 0 && lddy % 8 == 0 && ldx % 8 == 0 && lddw % 8 == 0 &&
                    dw_expert_stride % 8 == 0,
                XMA_ROCM_EUNSUPPORTED, "group_bwd_W: N_out=%d K_in=%d and leading dimensions must be multiples of 8",
                N_out, K_in);
    XMA_REQUIRE(lddy < ((int64_t)1 << 30) && ldx < ((int64_t)1 << 30) && lddy > 0 && ldx > 0, XMA_ROCM_EUNSUPPORTED,
                "group_bwd_W: leading dimensions must be below 2^30 elements");
    XMA_REQUIRE(DY && X && DW && expert_offsets && aligned16(DY) && aligned16(X) && aligned16(DW), XMA_ROCM_EINVAL,
                "group_bwd_W: null or misaligned operand");
    XMA_REQUIRE(sorted_scattered_idxs || (dy_grouped && x_grouped && !dy_scale), XMA_ROCM_EINVAL,
                "group_bwd_W: sorted_scattered_idxs is required unless everything is grouped");
    DwArgs a;
    a.DY = (const uint16_t *)DY;
    a.lddy = lddy;
    a.X = (const uint16_t *)X;
    a.ldx = ldx;
    a.scale = (const uint16_t *)dy_scale;
    a.idx = sorted_scattered_idxs;
    a.offs = expert_offsets;
    a.DW = (uint16_t *)DW;
    a.dw_es = dw_expert_stride;
    a.lddw = lddw;
    a.N_out = N_out;
    a.K_in = K_in;
    a.E = E;
    a.dy_grouped = dy_grouped;
    a.dy_fan_out = dy_fan_out;
    a.x_grouped = x_grouped;
    a.x_fan_out = x_fan_out;
    const int64_t grid = (int64_t)E * ((N_out + 255) / 256) * ((K_in + 255) / 256);
    XMA_REQUIRE(grid < ((int64_t)1 << 31), XMA_ROCM_EUNSUPPORTED, "group_bwd_W: grid too large");
    hipStream_t st = (hipStream_t)stream;
    a.dy_div = make_fastdiv((uint32_t)dy_fan_out);
    a.x_div = make_fastdiv((uint32_t)x_fan_out);
    if (dtype == XMA_ROCM_F32) return f32_group_bwd_W(a, M, st);
    if (dy_scale) return launch_dw_scaled(a, dtype, (int)grid, st);
    if (dtype == XMA_ROCM_BF16) return dispatch_dw<__bf16>(a, (int)grid, st);
    return grouped_dw_f16(a, (int)grid, st);
}

extern "C" int xma_rocm_group_bwd_W(const void *DY, int64_t lddy, int dy_grouped, int32_t dy_fan_out,
                                    const void *dy_scale, const void *X, int64_t ldx, int x_grouped, int32_t x_fan_out,
                                    const int64_t *sorted_scattered_idxs, const int64_t *expert_offsets, void *DW,
                                    int64_t dw_expert_stride, int64_t lddw, int32_t N_out, int32_t K_in, int32_t E,
                                    int dtype, void *stream) {
    return xma_group_bwd_W(DY, lddy, dy_grouped, dy_fan_out, dy_scale, X, ldx, x_grouped, x_fan_out, sorted_scattered_idxs, expert_offsets, DW,
                           dw_expert_stride, lddw, N_out, K_in, E, 0, dtype, stream);
}
#endif
