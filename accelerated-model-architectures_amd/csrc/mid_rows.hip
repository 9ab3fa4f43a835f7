// Grouped GEMMs for experts of some dozens to some hundreds of rows.  The 256 x 256 tiles of grouped_gemm.hip hold a compute unit
// to themselves: an expert of 260 rows pays for two of them, and between two tiles the matrix pipes idle for the epilogue, the
// next workgroup's dispatch and its chain of look-ups (offsets, row indices, first operands), which with few K steps, or with
// few rows behind a tile of dW, is as long as the K loop.  Here a tile is 128 x 256 and two workgroups share a compute unit, so
// that one multiplies while the other starts or stores.
//
// Workgroup = 4 wave64 (2 x 2), a wave owns 64 x 128 = 2 x 4 v_mfma_f32_32x32x16 blocks (128 fp32 accumulators per lane).  A K
// step of 64 is three items of 16 KB: Q (the 128 rows) and P0, P1 (two halves of the 256 columns: of every 128 the first and the
// second 64, so that a wave's columns are contiguous).  Two operand stages would take 96 KB; two workgroups have 80 KB each.  So
// the items go through a ring of five places in the order in which they are read, Q P0 P1 Q P0 ...: phase 1 of a step
// multiplies Q x P0, phase 2 Q x P1 with the fragments of Q still in registers, so Q and P0 are done with after phase 1 and P1
// after phase 2, and each freed place is filled at once:
//
//   barrier A(s)   Q(s), P0(s) have landed; every wave has read P1(s - 1)
//   phase 1        load P0(s + 1);                read Q(s), P0(s); 16 MFMAs per wave
//   barrier B(s)   P1(s) has landed; every wave has read Q(s), P0(s)
//   phase 2        load P1(s + 1), Q(s + 2);      read P1(s);       16 MFMAs per wave
//
// A load has a whole K step (two phases, 1024 cycles of the matrix pipe alone, twice that with both workgroups at work) to
// land; 2 x 40 KB are in flight per compute unit.  Each wave loads four 1 KB pieces of an item, so the waits are vmcnt(8): the
// two items behind the one that is waited for.  dW's sums run over an expert's rows from the first to the last, as in the 256 x 256
// kernels.  Forward types add in another order than those where the launch is cut into ranges of K (one fp32 sum per range, added in
// order), and where a column of tiles starts at a K step of its own (`turn`); both depend on the sizes only, not on the routing.
//
// Measured against the kernels that served these launches before (us; E experts, rows each): forward + backward GEMMs of E = 64, H =
// 2048, I = 1408, 96 rows 933 -> 715, 256 rows 1470 -> 1240; E = 128, H = 576, I = 256, 128 rows 197 -> 143; E = 8, H = 512, I =
// 1024, 256 rows 169 -> 95.  What bounds them: up to some 100 rows the stream of the weights, or of the stores of dW (4.5 to 5
// TB/s); beyond that the K loop, 2.1 us a step for the two workgroups of a compute unit (the products alone 0.9), part of it the
// board's power (cleared operands: 10 - 15 % shorter).  In launches of many rounds the 256 x 256 tiles, which move two thirds of the
// bytes per product through L2 and LDS, lead from about 350 (forward types) and 650 (dW) rows per expert on; in launches of a few
// rounds the smaller tiles stay ahead for longer, because they fill the last round better (mid_fwd_leads).
//
// Operand layouts in an item, as in grouped_gemm.hip with 16 KB instead of 32: K contiguous in memory [128 rows][8 chunks of
// 16 B], chunk c of row r at slot c ^ ((r >> 1) & 7); K the row index in memory [64 k-rows][16 chunks], chunk c of k-row kr at
// slot c ^ ((kr & 3) << 2), read with ds_read_b64_tr_b16.
#include <math.h>

#include "grouped_gemm_tile.hpp"
#include "mid_rows.hpp"

namespace xma_rocm {

namespace {

constexpr int MR_BM = 128, MR_BN = 256, MR_K = 64;
constexpr int MR_ITEM = MR_BM * MR_K * 2, MR_PLACES = 5, MR_SMEM_BYTES = MR_PLACES * MR_ITEM;
static_assert(4 * EPI_BWD_WAVE_BYTES <= MR_SMEM_BYTES && 4 * EPI_WAVE_BYTES <= MR_SMEM_BYTES, "epilogue staging fits into the ring");
constexpr int MR_RUN = 512; // workgroups that run at the same time on a 256-CU device
constexpr int MR_SMEM_ALONE = MR_SMEM_BYTES + 1024; // too much for two workgroups of a compute unit
constexpr int MR_MAX_E = 1024;
constexpr int MR_TURN_ROWS = 144; // rows per expert up to which the tiles of a column start at a K step of their own

// Every item this wave has loaded has landed but for the youngest `n` pieces, and its LDS reads have returned; then meet the others.
#define MR_WAIT_AND_BARRIER(n) asm volatile("s_waitcnt vmcnt(" #n ") lgkmcnt(0)\n\ts_barrier" ::: "memory")

// A dword at base + off; in flight until mr_wait_idx_and_barrier, which leaves the four youngest pieces in flight.
__device__ __forceinline__ void mr_load_dword(uint32_t &dst, const void *base, uint32_t off) {
    asm volatile("global_load_dword %0, %1, %2" : "=v"(dst) : "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void mr_wait_idx_and_barrier(uint32_t (&v)[4]) {
    asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory");
}

// Workgroup id -> tile of the launch's `total`, or -1.  Ids go to the 8 XCDs round-robin; of every run of 512 tiles, and of the
// shorter last one, each XCD gets one contiguous eighth, whose tiles share operand panels in its L2.  Ids up to total + 7 are used.
__device__ __forceinline__ int mr_tile_of(int w, int total) {
    const int full = total / MR_RUN * MR_RUN;
    if (w < full) {
        const int x = w & (MR_RUN - 1);
        return (w - x) + (x & 7) * (MR_RUN / 8) + (x >> 3);
    }
    const int t = total - full, c = (t + 7) >> 3, v = w - full, l = (v & 7) * c + (v >> 3);
    return ((v >> 3) < c && l < t) ? full + l : -1;
}

__device__ __forceinline__ int mr_wave_scan(int v, int lane) { // inclusive
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int t = __shfl_up(v, d);
        if (lane >= d) v += t;
    }
    return v;
}

// ---- fragments of an item; blk: 32-row (or column) block behind R0, which is a multiple of 64
template <int TR> struct ItemFrag {
    uint32_t off[4]; // K contiguous: one per k16 slice; transposed: one per block
};
template <int TR> __device__ __forceinline__ void mr_make_frag(ItemFrag<TR> &f, int R0, int lane) {
    if constexpr (TR == 0) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) f.off[kk] = (uint32_t)((R0 + (lane & 31)) * 128 + (((2 * kk + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4));
    } else {
        const int p = lane & 15, G = lane >> 4, kr = ((G >> 1) << 3) + (p >> 2);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int m = R0 + 32 * b + ((G & 1) << 4) + ((p & 3) << 2);
            f.off[b] = (uint32_t)(kr * 256 + (((m >> 3) ^ ((kr & 3) << 2)) << 4) + ((m & 7) << 1));
        }
    }
}
template <int TR> __device__ __forceinline__ u32x4 mr_read_frag(const unsigned char *item, const ItemFrag<TR> &f, int blk, int kk) {
    if constexpr (TR == 0) {
        return *(const u32x4 *)(item + f.off[kk] + blk * 4096);
    } else {
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) v4s *lds_v4s;
        const unsigned char *at = item + f.off[blk] + kk * 4096;
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)at));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(at + 1024)));
        return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
}

// Places of the ring as byte offsets; the items of a step lie in three consecutive ones.
__device__ __forceinline__ uint32_t mr_place_after(uint32_t place, int n) {
    const uint32_t p = place + (uint32_t)(n * MR_ITEM);
    return p >= (uint32_t)MR_SMEM_BYTES ? p - MR_SMEM_BYTES : p;
}

// The K loop over steps 0 .. steps - 1 (> 0).  load(IC<0 | 1 | 2>, step, place) issues this wave's four pieces of Q, P0 or P1;
// Q(0), P0(0), P1(0) and, with more than one step, Q(1) are under way, in the place `at` and those behind it.  begin(s) and mid(s) stand
// in front of the loads of phase 1 and behind those of P1 in phase 2 (the row indices of a gathered operand); wait_b() is the wait and
// barrier B of a step with another one behind it.  NB: 32-row blocks of this wave's 64 rows that hold valid rows.
template <typename T, int QTR, int PTR, int NB, typename Load, typename Begin, typename WaitB, typename Mid>
__device__ __forceinline__ void mr_k_loop(f32x16 (&acc)[4][2], const unsigned char *smem, const ItemFrag<QTR> &qf,
                                          const ItemFrag<PTR> &pf, int steps, uint32_t at, Load load, Begin begin,
                                          WaitB wait_b, Mid mid) {
    u32x4 q[4][2];
    auto phase = [&](uint32_t place, auto HALF) {
        const unsigned char *item = smem + place;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            if constexpr (HALF.value == 0) {
#pragma unroll
                for (int i = 0; i < NB; ++i) q[kk][i] = mr_read_frag<QTR>(smem + at, qf, i, kk);
            }
#pragma unroll
            for (int b = 0; b < (NB ? 2 : 0); ++b) {
                const u32x4 p = mr_read_frag<PTR>(item, pf, b, kk);
#pragma unroll
                for (int i = 0; i < NB; ++i) acc[2 * HALF.value + b][i] = Elem<T>::mfma(p, q[kk][i], acc[2 * HALF.value + b][i]);
            }
        }
    };
    for (int s = 0; s + 1 < steps; ++s) {
        MR_WAIT_AND_BARRIER(8);
        begin(s);
        load(IC<1>{}, s + 1, mr_place_after(at, 4));
        phase(mr_place_after(at, 1), IC<0>{});
        wait_b();
        load(IC<2>{}, s + 1, at);
        mid(s);
        if (s + 2 < steps) load(IC<0>{}, s + 2, mr_place_after(at, 1));
        phase(mr_place_after(at, 2), IC<1>{});
        at = mr_place_after(at, 3);
    }
    MR_WAIT_AND_BARRIER(4);
    phase(mr_place_after(at, 1), IC<0>{});
    MR_WAIT_AND_BARRIER(0);
    phase(mr_place_after(at, 2), IC<1>{});
    MR_WAIT_AND_BARRIER(0); // the ring is free for the epilogue
}

// ------------------------------------------------------------------------------------------------
// forward / dX: Q = activation rows, P = weight rows (WT = 0, W[e] is (N, K)) or columns (WT = 1, W[e] is (K, N))
// ------------------------------------------------------------------------------------------------
struct MidTile {
    int e, n0, row0, rows_valid, part;
};

// Which of the launch's tiles x K ranges workgroup w computes: expert-major, rows first, all tiles of a K range before the next.
// Every wave scans the experts in registers, 64 at a time (lane = expert): no LDS, no barrier.  false: none is left.
__device__ __forceinline__ bool mr_locate(const FwdArgs &a, int w, int parts, int lane, MidTile &t) {
    const int NT = (a.N + MR_BN - 1) / MR_BN;
    auto tiles = [&](int x, int &lo, int &rows) {
        lo = rows = 0;
        if (x < a.E) {
            const int hi = (int)a.offs[x];
            lo = x ? (int)a.offs[x - 1] : 0;
            rows = hi - lo;
        }
        return (rows + MR_BM - 1) / MR_BM * NT;
    };
    int lo, rows, s = mr_wave_scan(tiles(lane, lo, rows), lane), total = __builtin_amdgcn_readlane(s, WAVE - 1);
    if (a.E > WAVE) {
        int sum = 0;
        for (int b = WAVE; b < a.E; b += WAVE) {
            int l, r;
            sum += tiles(b + lane, l, r);
        }
        total += __builtin_amdgcn_readlane(mr_wave_scan(sum, lane), WAVE - 1);
    }
    const int u = mr_tile_of(w, total * parts);
    if (u < 0) return false;
    t.part = u / total;
    const int L = u - t.part * total;
    int base = 0, before = 0; // first expert of the chunk, tiles in front of it
    while (before + __builtin_amdgcn_readlane(s, WAVE - 1) <= L) { // L < total: ends at the chunk that holds it
        before += __builtin_amdgcn_readlane(s, WAVE - 1);
        base += WAVE;
        s = mr_wave_scan(tiles(base + lane, lo, rows), lane);
    }
    const int in_chunk = L - before;
    const int at = __builtin_ctzll(__ballot(s > in_chunk)); // the first expert whose tiles reach beyond L
    const int row_lo = __builtin_amdgcn_readlane(lo, at), n = __builtin_amdgcn_readlane(rows, at), tiles_m = (n + MR_BM - 1) / MR_BM;
    const int local = in_chunk - (__builtin_amdgcn_readlane(s, at) - tiles_m * NT), col = local / tiles_m, m = local - col * tiles_m;
    t.e = base + at;
    t.n0 = col * MR_BN;
    t.row0 = row_lo + m * MR_BM;
    t.rows_valid = n - m * MR_BM < MR_BM ? n - m * MR_BM : MR_BM;
    return true;
}

// EPI = -1: the launch is cut along K, `parts` ranges of steps_per steps; the fp32 sums go to sums[range][M][N].
// One workgroup per tile: the hardware hands out the next one where one has ended, which suits tiles that take from a third (few
// rows) to a whole of the longest.  (512 workgroups that walk the tiles and fetch the next one's indices and first operands
// ahead were 5 - 12 % slower.)
template <typename T, int WT, int EPI>
__global__ __launch_bounds__(GEMM_THREADS, 2) void mid_fwd_kernel(const FwdArgs a, float *__restrict__ sums, int parts, int steps_per) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    MidTile t;
    if (!mr_locate(a, blockIdx.x, EPI < 0 ? parts : 1, lane, t)) return; // uniform
    const int KT = (a.K + MR_K - 1) / MR_K;
    const int s_begin = EPI < 0 ? t.part * steps_per : 0;
    const int steps = (EPI < 0 && s_begin + steps_per < KT ? s_begin + steps_per : KT) - s_begin; // > 0: the host cuts no empty range
    const int wq = (wave & 1) * 64, wp = (wave >> 1) * 128;
    auto clamp_row = [&](int r) { return r < t.rows_valid ? r : t.rows_valid - 1; };

    // rows of this lane's pieces of Q, and of its part of the epilogue
    uint32_t q_off[4], p_off[2][4];
    EpiRows er;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = clamp_row(32 * wave + 8 * i + (lane >> 3));
        const uint32_t src = a.x_grouped ? (uint32_t)r : fastdiv((uint32_t)a.idx[t.row0 + r], a.fan_div);
        q_off[i] = mul_add_u32(src, (uint32_t)(2 * a.ldx), (uint32_t)((lane & 7) ^ (((i & 1) << 2) + (lane >> 4))) * 16);
    }
    if constexpr (EPI >= 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            er.idx[i] = 0, er.sc[i] = 1.f;
            if (!a.y_grouped || a.scale) er.idx[i] = (int)a.idx[t.row0 + clamp_row(wq + 32 * i + (lane & 31))];
        }
        if (a.scale) {
#pragma unroll
            for (int i = 0; i < 2; ++i) er.sc[i] = Elem<T>::lo((uint32_t)a.scale[er.idx[i]]);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (WT == 0) {
                const int r = 32 * wave + 8 * i + (lane >> 3); // row of the item: 64 columns of either 128
                int col = (r >> 6) * 128 + h * 64 + (r & 63);
                if (t.n0 + col >= a.N) col = a.N - 1 - t.n0; // computed and never stored
                p_off[h][i] = mul_add_u32((uint32_t)col, (uint32_t)(2 * a.ldw), (uint32_t)((lane & 7) ^ (((i & 1) << 2) + (lane >> 4))) * 16);
            } else {
                const int c = (lane & 15) ^ ((lane >> 4) << 2); // chunk of the item
                int chunk = (c >> 3) * 16 + h * 8 + (c & 7);
                const int max_chunk = ((a.N - t.n0) >> 3) - 1;
                if (chunk > max_chunk) chunk = max_chunk;
                p_off[h][i] = mul_add_u32((uint32_t)(16 * wave + 4 * i + (lane >> 4)), (uint32_t)(2 * a.ldw), (uint32_t)chunk * 16);
            }
        }
    const uint16_t *q_base = a.x_grouped ? a.X + (int64_t)t.row0 * a.ldx : a.X;
    const uint16_t *p_base = a.W + (int64_t)t.e * a.w_es + (WT == 0 ? (int64_t)t.n0 * a.ldw : (int64_t)t.n0);
    const uint32_t lds0 = lds_addr_of(smem) + (uint32_t)wave * 4096;
    const int k_left = a.K - (KT - 1) * MR_K; // of the last step
    // W as (N, K): workgroups that run at the same time are at about the same step, and with all of them walking K from the front
    // their requests of a moment would fall on the same 128 bytes of every row of W, a fraction of the memory channels where the
    // row pitch is a multiple of 4 KB.  So the tiles of every column of tiles start at a step of their own and wrap around,
    // while most experts have one tile of rows (tiles that share activations drift apart by it): 64 rows for each of 8 experts,
    // H = 2048, I = 8192, up-projection 134 -> 108 us; 192 rows, H = 4096, I = 14336, 520 -> 584.
    const int turn = WT == 0 && a.M <= (int64_t)MR_TURN_ROWS * a.E ? (t.n0 / MR_BN * 5 + t.e * 3) % steps : 0;
    auto load = [&](auto ITEM, int s, uint32_t place) {
        constexpr int item = ITEM.value;
        if constexpr (WT == 0) s = s + turn < steps ? s + turn : s + turn - steps;
        s += s_begin;
        const int64_t step = (item == 0 || WT == 0) ? MR_K : (int64_t)MR_K * a.ldw;
        const i32x4 desc = buf_desc((item == 0 ? q_base : p_base) + s * step);
        const bool cut = k_left < MR_K && s == KT - 1; // uniform: chunks past K are asked for outside the buffer and read zeros
        static_for<4>([&](auto I) {
            constexpr int i = I.value;
            uint32_t off = item == 0 ? q_off[i] : p_off[item == 2 ? 1 : 0][i];
            if (cut) {
                const int k = (item == 0 || WT == 0) ? ((lane & 7) ^ (((i & 1) << 2) + (lane >> 4))) * 8 : 16 * wave + 4 * i + (lane >> 4);
                off = k < k_left ? off : BUF_OUTSIDE;
            }
            lds_dma16_buf(desc, off, (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + place)), i * 1024);
        });
    };
    load(IC<0>{}, 0, 0);
    load(IC<1>{}, 0, MR_ITEM);
    load(IC<2>{}, 0, 2 * MR_ITEM);
    if (steps > 1) load(IC<0>{}, 1, 3 * MR_ITEM);

    f32x16 acc[4][2];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int c = 0; c < 16; ++c) acc[j][i][c] = 0.f;
    if constexpr (EPI >= 0) {
        if (a.bias) { // the first term of every sum, as a product with ones (see add_bias in grouped_gemm.hip)
            const uint16_t *b = a.bias + (int64_t)t.e * a.bias_es;
            const bool k0 = lane < 32;
            const u32x4 ones = {k0 ? one_bits<T>() : 0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int col = t.n0 + wp + 32 * j + (lane & 31);
                if (col >= a.N) col = a.N - 1;
                const uint32_t v = b[col];
                const u32x4 p = {k0 ? v : 0u, 0u, 0u, 0u};
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[j][i] = Elem<T>::mfma(p, ones, acc[j][i]);
            }
        }
    }
    ItemFrag<0> qf;
    ItemFrag<WT> pf;
    mr_make_frag<0>(qf, wq, lane);
    mr_make_frag<WT>(pf, wp >> 1, lane);
    auto nothing = [](int) {};
    auto wait_b = []() { MR_WAIT_AND_BARRIER(8); };
    const int rows_left = t.rows_valid - wq;
    if (rows_left > 32)
        mr_k_loop<T, 0, WT, 2>(acc, smem, qf, pf, steps, 0, load, nothing, wait_b, nothing);
    else if (rows_left > 0)
        mr_k_loop<T, 0, WT, 1>(acc, smem, qf, pf, steps, 0, load, nothing, wait_b, nothing);
    else
        mr_k_loop<T, 0, WT, 0>(acc, smem, qf, pf, steps, 0, load, nothing, wait_b, nothing);

    if constexpr (EPI >= 0) {
        tile_epilogue<T, EPI, 2>(a, acc, smem, t.row0, t.rows_valid, t.n0, tid, -1, &er);
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = wq + 32 * i + (lane & 31);
            if (r >= t.rows_valid) continue;
            float *mine = sums + ((int64_t)t.part * a.M + t.row0 + r) * a.N;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int n = t.n0 + wp + 32 * j + 8 * g + 4 * (lane >> 5);
                    if (n < a.N) *(float4 *)(mine + n) = make_float4(acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]);
                }
        }
    }
}

// ------------------------------------------------------------------------------------------------
// dW[e][o][i] = sum over the expert's rows n of DY[n][o] X[n][i]: Q = dY columns, P = X columns, K = the expert's rows, 64 at a
// time, zeros beyond the last.  GQ / GP = 1: the rows of dY / X are taken through sorted_scattered_idxs (index / fan_out).
// ------------------------------------------------------------------------------------------------
constexpr int MR_DW_BAND = 8; // tile rows of a band: the 64 tiles an XCD works on are 8 x 8, 1024 columns of dY x 2048 of X

struct MidDwTile {
    int e, o0, i0, rows;
    int64_t row_lo;
};

// NT = 1: the rows of dW go past L2 (a variant of its own: the compiler merges the two kinds of store into one where a branch picks).
template <typename T, int GQ, int GP, int NT>
__global__ __launch_bounds__(GEMM_THREADS, 2) void mid_dw_kernel(const DwArgs a) {
    constexpr bool GATHER = GQ != 0 || GP != 0;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int OT = (a.N_out + MR_BM - 1) / MR_BM, IT = (a.K_in + MR_BN - 1) / MR_BN, total = a.E * OT * IT;
    const int wq = (wave & 1) * 64, wp = (wave >> 1) * 128;
    const int c = (lane & 15) ^ ((lane >> 4) << 2); // this lane's chunk of an item
    const int kr0 = 16 * wave + (lane >> 4);        // k-row of piece i: kr0 + 4 i
    const uint32_t lddy_b = (uint32_t)a.lddy * 2, ldx_b = (uint32_t)a.ldx * 2;
    const uint32_t lds0 = lds_addr_of(smem) + (uint32_t)wave * 4096;
    ItemFrag<1> qf, pf;
    mr_make_frag<1>(qf, wq, lane);
    mr_make_frag<1>(pf, wp >> 1, lane);

    // Up to 64 experts wait in registers (lane = expert), ranked by decreasing row count: the longest K loops start first (see
    // grouped_gemm_dw_kernel).  Beyond that the order is that of the index, and a tile's offsets come from memory.
    int lo32 = 0, cnt = -1, rank = 0;
    if (a.E <= WAVE) {
        const int hi = (int)a.offs[lane < a.E ? lane : a.E - 1];
        lo32 = __shfl_up(hi, 1);
        if (lane == 0) lo32 = 0;
        if (lane < a.E) cnt = hi - lo32;
        for (int i = 0; i < a.E; ++i) {
            const int ci = __builtin_amdgcn_readlane(cnt, i);
            rank += (ci > cnt || (ci == cnt && i < lane)) ? 1 : 0;
        }
    }
    auto find = [&](int w, MidDwTile &t) -> bool {
        const int L = mr_tile_of(w, total);
        if (L < 0) return false;
        const int r = L / (OT * IT), rem = L - r * (OT * IT);
        if (a.E <= WAVE) {
            t.e = __builtin_ctzll(__ballot(rank == r && lane < a.E)); // exactly one lane
            t.row_lo = __builtin_amdgcn_readlane(lo32, t.e);
            t.rows = __builtin_amdgcn_readlane(cnt, t.e);
        } else {
            t.e = r;
            t.row_lo = r ? a.offs[r - 1] : 0;
            t.rows = (int)(a.offs[r] - t.row_lo);
        }
        const int band = rem / (MR_DW_BAND * IT), in_band = rem - band * (MR_DW_BAND * IT);
        const int band_rows = (OT - band * MR_DW_BAND < MR_DW_BAND) ? OT - band * MR_DW_BAND : MR_DW_BAND;
        const int col = in_band / band_rows;
        t.o0 = (band * MR_DW_BAND + in_band - col * band_rows) * MR_BM;
        t.i0 = col * MR_BN;
        return true;
    };

    // Rows of a step: byte offsets of this lane's four pieces, of the step that is loaded next for a gathered operand, of every step
    // relative to its first row for a grouped one; columns past the edge of dW are clamped.  All of the tile that is loaded.
    MidDwTile cur;
    const uint16_t *q_base = nullptr, *p_base = nullptr;
    const int64_t *idx = nullptr;
    uint32_t q_col = 0, p_col[2] = {0, 0}, q_row[4], p_row[4], idx_next[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q_row[i] = (uint32_t)(kr0 + 4 * i) * lddy_b, p_row[i] = (uint32_t)(kr0 + 4 * i) * ldx_b;
    auto set_tile = [&]() {
        const int q_max = ((a.N_out - cur.o0) >> 3) - 1, p_max = ((a.K_in - cur.i0) >> 3) - 1;
        q_col = (uint32_t)(c < q_max ? c : q_max) * 16;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int ch = (c >> 3) * 16 + h * 8 + (c & 7);
            p_col[h] = (uint32_t)(ch < p_max ? ch : p_max) * 16;
        }
        q_base = a.DY + cur.o0 + (GQ ? 0 : cur.row_lo * a.lddy);
        p_base = a.X + cur.i0 + (GP ? 0 : cur.row_lo * a.ldx);
        idx = a.idx + cur.row_lo;
    };
    auto from_idx = [&](const uint32_t (&v)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (GQ) q_row[i] = fastdiv(v[i], a.dy_div) * lddy_b;
            if (GP) p_row[i] = fastdiv(v[i], a.x_div) * ldx_b;
        }
    };
    auto load = [&](auto ITEM, int s, uint32_t place) {
        constexpr int item = ITEM.value, gathered = item == 0 ? GQ : GP;
        const uint16_t *base = item == 0 ? q_base : p_base;
        const i32x4 desc = buf_desc(gathered ? base : base + (int64_t)s * MR_K * (item == 0 ? a.lddy : a.ldx));
        const int left = cur.rows - s * MR_K;
        static_for<4>([&](auto I) {
            constexpr int i = I.value;
            uint32_t off = item == 0 ? q_row[i] + q_col : p_row[i] + p_col[item == 2 ? 1 : 0];
            if (left < MR_K) off = kr0 + 4 * i < left ? off : BUF_OUTSIDE; // rows past the expert's last read zeros
            lds_dma16_buf(desc, off, (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + place)), i * 1024);
        });
    };
    // the indices of the first two steps of a tile, one tile ahead
    uint32_t idx0[4] = {0u, 0u, 0u, 0u}, idx1[4] = {0u, 0u, 0u, 0u};
    auto fetch_idx = [&](const MidDwTile &t) {
        if (!GATHER || t.rows == 0) return; // uniform
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r0 = kr0 + 4 * i, r1 = MR_K + r0;
            idx0[i] = (uint32_t)a.idx[t.row_lo + (r0 < t.rows ? r0 : t.rows - 1)];
            idx1[i] = (uint32_t)a.idx[t.row_lo + (r1 < t.rows ? r1 : t.rows - 1)];
        }
    };
    // The first four items of a tile, in the places 1 to 4; place 0 stays free for the staging of the tile before it.
    auto first_items = [&]() {
        if (cur.rows == 0) return; // uniform
        if constexpr (GATHER) from_idx(idx0);
        load(IC<0>{}, 0, MR_ITEM);
        load(IC<1>{}, 0, 2 * MR_ITEM);
        load(IC<2>{}, 0, 3 * MR_ITEM);
        if constexpr (GATHER) from_idx(idx1);
        if (cur.rows > MR_K) load(IC<0>{}, 1, 4 * MR_ITEM);
    };
    int w = blockIdx.x;
    if (!find(w, cur)) return; // uniform
    fetch_idx(cur);
    set_tile();
    first_items();
    for (bool more = true; more;) {
        f32x16 acc[4][2];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;
        w += MR_RUN;
        MidDwTile nxt;
        more = find(w, nxt);
        if (more) fetch_idx(nxt); // waited for behind the K loop
        if (cur.rows > 0) {
            // Indices of step s + 2 (low dwords): requested in front of phase 1's loads, waited for at barrier B - the four
            // pieces of P0 are younger - and used for Q in phase 2 and for P one step later.  The loads are inline assembly: for
            // a load of its own the compiler would wait by draining every piece in flight, which it does not know of.
            auto begin = [&](int s) {
                if constexpr (GATHER) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = (s + 2) * MR_K + kr0 + 4 * i;
                        mr_load_dword(idx_next[i], idx, (uint32_t)(r < cur.rows ? r : cur.rows - 1) * 8);
                    }
                }
            };
            auto wait_b = [&]() {
                if constexpr (GATHER)
                    mr_wait_idx_and_barrier(idx_next);
                else
                    MR_WAIT_AND_BARRIER(8);
            };
            auto mid = [&](int) {
                if constexpr (GATHER) from_idx(idx_next);
            };
            mr_k_loop<T, 1, 1, 2>(acc, smem, qf, pf, (cur.rows + MR_K - 1) / MR_K, MR_ITEM, load, begin, wait_b, mid);
        }
        const MidDwTile done = cur;
        if (more) {
            cur = nxt;
            set_tile();
            first_items();
        }
        // a 32-row block x 64 columns at a time through 4 KB of place 0 that belong to the wave, out as rows of 128 bytes: past L2 (NT)
        // where they start on 64-byte boundaries; elsewhere most lines come from two stores, which L2 has to join (40 experts of
        // 3864 x 8136, 46 rows each: 1640 us past it, 990 through it; on the boundaries, 129 to 640 rows, 0.71 against 0.78 of the time of
        // the 256 x 256 tiles)
        const int lrow = lane & 31, lhalf = lane >> 5;
        uint16_t *DWe = a.DW + (int64_t)done.e * a.dw_es;
        unsigned char *stage = smem + wave * 4096;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int obase = done.o0 + wq + i * 32;
            if (obase >= a.N_out) break; // wave-uniform
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const f32x16 &v = acc[2 * h + j][i];
                        *(u32x2 *)(stage + lrow * 128 + (((4 * j + g) ^ ((lrow >> 1) & 7)) << 4) + 8 * lhalf) =
                            u32x2{Elem<T>::pack(v[4 * g], v[4 * g + 1]), Elem<T>::pack(v[4 * g + 2], v[4 * g + 3])};
                    }
                wave_lds_sync();
                const int cz = done.i0 + wp + h * 64 + (lane & 7) * 8;
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const int r = 8 * it + (lane >> 3), o = obase + r;
                    const u32x4 v = *(const u32x4 *)(stage + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4));
                    if (o < a.N_out && cz < a.K_in) {
                        u32x4 *at = (u32x4 *)(DWe + (int64_t)o * a.lddw + cz);
                        if constexpr (NT != 0)
                            __builtin_nontemporal_store(v, at);
                        else
                            *at = v;
                    }
                }
                wave_lds_sync(); // the next block overwrites the area
            }
        }
    }
}

// Tiles of `height` rows x 256 columns that the offsets will give, about: one per expert while nearly all fit into it, half a tile
// of an expert's last rows beyond that.
inline double tiles_about(int64_t M, int N, int E, int height) {
    const double rows = (double)M / E;
    return (rows + 2.5 * sqrt(rows) <= height ? (M < E ? M : E) : E * (rows / height + 0.5)) * ((N + MR_BN - 1) / MR_BN);
}

// The length of a forward-type launch of 128 x 256 tiles cut into S ranges of K, about, and the S (each at least 4 steps) that makes
// it shortest.  t workgroups on 256 compute units stream their operands at 4.9 TB/s from about 185 busy units on; alone on its unit a
// workgroup takes 1.1 us a step, two that share one 2.1 us each, with 512 at a time, 2.4 where more wait behind them (power); the
// sums of S > 1 ranges go through memory twice (3.3 TB/s) behind one more launch.  This and tiles256_seconds were fitted together to 336
// measured pairs of launches (the layers of the benchmark and six others, 100 to 4000 rows per expert): within 12 and 10 % on average.
// Of the 25,500 other pairs in mid_fwd_leads that takes 17,600 launches, which are 1.46 times as fast as the 256 x 256 ones on geometric
// average; one in thirty of them is more than 3 % slower, the worst takes 1.59 times as long (64 experts of 98 rows, K = 16640).
inline double mid_fwd_seconds(int64_t M, int N, int K, int E, int epilogue, int *best) {
    // Long K: one tile too many for a round of K ranges is another round of long ones (8 experts of H = 1024, K = 16384, 270 rows, where
    // most need a third tile: 174 us in 6 ranges, 148 now), so the tiles that experts of average rows need are counted in full.
    const double rows = (double)M / E, whole = E * ceil((rows - sqrt(rows) / 2) / MR_BM) * ((N + MR_BN - 1) / MR_BN);
    const double some = tiles_about(M, N, E, MR_BM), tiles = K > 8192 && whole > some ? whole : some, bytes = 2.0 * (M < E ? M : E) * N * K + 2.0 * M * (N + K);
    const double epi = epilogue == XMA_ROCM_EPI_SWIGLU_BWD ? 7.7e-6 : 0.;
    const int steps = (K + MR_K - 1) / MR_K;
    double shortest = 1e30;
    *best = 1;
    for (int S = 1; S <= 8 && (S == 1 || (steps / S >= 4 && (double)S * M * N * 4 <= 256e6)); ++S) {
        const double t = tiles * S, rounds = t / MR_RUN, busy = t <= MR_RUN / 2 ? t : t < MR_RUN ? t / 2 : MR_RUN / 2;
        const double stream = bytes / 4.9e12 * (busy < 185 ? 185 / busy : 1.);
        const double step = rounds <= 0.5 ? 1.1e-6 : rounds <= 1 ? 2.1e-6 * (0.5 + rounds / 2) : 2.4e-6 * rounds;
        const double walk = ((steps + S - 1) / S) * step + (S == 1 ? epi * (rounds > 1 ? rounds : 1.) : 0.);
        const double time = pow(pow(stream, 4.4) + pow(walk, 4.4), 1 / 4.4) + 7e-6 + (S > 1 ? 8.0 * S * M * N / 3.3e12 + 4e-6 : 0.);
        if (time < shortest) shortest = time, *best = S;
    }
    return shortest;
}

inline int mid_fwd_splits(int64_t M, int N, int K, int E) {
    int S;
    mid_fwd_seconds(M, N, K, E, XMA_ROCM_EPI_STORE, &S);
    return S;
}

// The same for the 256 x 256 kernels: 1.6 us a step, 8 to 21 us at a tile's edges by its epilogue, in rounds of 256 tiles; a last round
// is a round to itself in a launch of up to three, a third of one behind more; its tiles run as K slices where they are few enough
// for two or more slices each (two more launches, sums through memory).
inline double tiles256_seconds(int64_t M, int N, int K, int E, int epilogue) {
    const double tiles = tiles_about(M, N, E, 256), n = tiles / 256, full = floor(n), rest = tiles - 256 * full;
    const int steps = (K + MR_K - 1) / MR_K;
    const double bytes = 2.0 * (M < E ? M : E) * N * K + 2.0 * M * (N + K);
    const double edges = epilogue == XMA_ROCM_EPI_SWIGLU_BWD ? 20.8e-6 : epilogue == XMA_ROCM_EPI_SWIGLU ? 10.6e-6 : 7.6e-6;
    const int parts = rest > 0 ? (int)(256 / rest < steps / 8 ? 256 / rest : steps / 8) : 0;
    const bool split = parts >= 2 && tiles <= 12 * 256;
    double rounds = full + (rest <= 0 ? 0. : split ? 1. / parts : 1.);
    if (n > 3 && rounds > n + 0.34) rounds = n + 0.34;
    const double walk = rounds * (steps * 1.6e-6 * (n < 1 ? 0.9 + 0.1 * n : 1.) + edges);
    return pow(pow(walk, 3.2) + pow(bytes / 4.5e12, 3.2), 1 / 3.2) + (split ? rest * parts * 2 * 262144 / 3.5e12 : 0.) + (steps >= 16 ? 10e-6 : 0.);
}

template <typename T, int WT, int EPI> int mid_launch_fwd(const FwdArgs &a, float *sums, hipStream_t st) {
    const int KT = (a.K + MR_K - 1) / MR_K;
    const int S_max = sums ? mid_fwd_splits(a.M, a.N, a.K, a.E) : 1, steps_per = (KT + S_max - 1) / S_max;
    const int S = (KT + steps_per - 1) / steps_per;
    const int64_t grid = (a.M / MR_BM + a.E) * ((a.N + MR_BN - 1) / MR_BN) * S + 7; // at most
    // The dispatcher puts two neighbouring workgroups of an XCD on one compute unit while others have none.  A launch that leaves
    // compute units idle asks for more LDS than half a compute unit has, and gets one of its own for every workgroup.
    const int smem = tiles_about(a.M, a.N, a.E, MR_BM) * S <= MR_RUN / 2 ? MR_SMEM_ALONE : MR_SMEM_BYTES;
    int rc;
    if (S == 1) {
        if ((rc = gemm_set_smem(mid_fwd_kernel<T, WT, EPI>, MR_SMEM_ALONE))) return rc;
        mid_fwd_kernel<T, WT, EPI><<<(unsigned)grid, GEMM_THREADS, smem, st>>>(a, nullptr, 1, KT);
        return xma_check_launch("mid_fwd_kernel");
    }
    if ((rc = gemm_set_smem(mid_fwd_kernel<T, WT, -1>, MR_SMEM_ALONE))) return rc;
    mid_fwd_kernel<T, WT, -1><<<(unsigned)grid, GEMM_THREADS, smem, st>>>(a, sums, S, steps_per);
    if ((rc = xma_check_launch("mid_fwd_kernel (K ranges)"))) return rc;
    return split_sums_epilogue(a, sums, S, EPI == EPI_SWIGLU_BWD_SCALED_ACT ? (int)XMA_ROCM_EPI_SWIGLU_BWD : EPI,
                               __is_same(T, __bf16) ? XMA_ROCM_BF16 : XMA_ROCM_F16, st);
}

template <typename T, int WT> int mid_dispatch_fwd(const FwdArgs &a, int epi, float *part, hipStream_t st) {
    if (epi == XMA_ROCM_EPI_STORE) return mid_launch_fwd<T, WT, XMA_ROCM_EPI_STORE>(a, part, st);
    if (epi == XMA_ROCM_EPI_SWIGLU) return mid_launch_fwd<T, WT, XMA_ROCM_EPI_SWIGLU>(a, part, st);
    if (epi == (WT ? EPI_GELU_BWD : EPI_GELU)) return mid_launch_fwd<T, WT, WT ? EPI_GELU_BWD : EPI_GELU>(a, part, st);
    if (a.aux2) return mid_launch_fwd<T, WT, EPI_SWIGLU_BWD_SCALED_ACT>(a, part, st);
    return mid_launch_fwd<T, WT, XMA_ROCM_EPI_SWIGLU_BWD>(a, part, st);
}

// whether the 128-byte pieces of dW's rows start on 64-byte boundaries
inline int mr_whole_lines(const DwArgs &a) { return (((uintptr_t)a.DW | (uintptr_t)(a.lddw * 2) | (uintptr_t)(a.dw_es * 2)) & 63) == 0; }

template <typename T, int GQ, int GP, int NT> int mid_launch_dw(const DwArgs &a, hipStream_t st) {
    const int64_t tiles = (int64_t)a.E * ((a.N_out + MR_BM - 1) / MR_BM) * ((a.K_in + MR_BN - 1) / MR_BN);
    const int rc = gemm_set_smem(mid_dw_kernel<T, GQ, GP, NT>, MR_SMEM_BYTES);
    if (rc) return rc;
    mid_dw_kernel<T, GQ, GP, NT><<<(unsigned)(tiles + 7 < MR_RUN ? tiles + 7 : MR_RUN), GEMM_THREADS, MR_SMEM_BYTES, st>>>(a);
    return xma_check_launch("mid_dw_kernel");
}

template <typename T, int NT> int mid_dispatch_dw(const DwArgs &a, hipStream_t st) {
    if (!a.dy_grouped) return mid_launch_dw<T, 1, 0, NT>(a, st);
    return a.x_grouped ? mid_launch_dw<T, 0, 0, NT>(a, st) : mid_launch_dw<T, 0, 1, NT>(a, st);
}

} // namespace

size_t mid_fwd_workspace_bytes(int64_t M, int32_t N, int32_t K, int32_t E) {
    const int S = mid_fwd_splits(M, N, K, E);
    return S == 1 ? 0 : (size_t)S * (size_t)M * (size_t)N * sizeof(float);
}

bool mid_fwd_has(int64_t M, int32_t E, int wt, int epi) {
    // GELU comes in the layouts that the layer launches, x @ W^T and dy @ W.  SwiGLU also in the other two (weights stored
    // transposed): streaming the weights once per 32 rows instead costs them, 8 experts of H = 2048, I = 8192, 96 rows each,
    // W1 as (H, 2I), 351 us against 116, W2 as (I, H) 167 against 57.
    return M > 0 && M <= 65535 && E <= MR_MAX_E && !(epi == EPI_GELU && wt) && !(epi == EPI_GELU_BWD && !wt);
}

bool mid_fwd_takes(const FwdArgs &a, int wt, int epi) {
    const int64_t x_rows = a.x_grouped ? MR_BM : (a.M + a.fan_out - 1) / a.fan_out; // 32-bit byte offsets from a tile's base
    return mid_fwd_has(a.M, a.E, wt, epi) && x_rows * a.ldx * 2 < ((int64_t)1 << 32) && (int64_t)MR_BN * a.ldw * 2 < ((int64_t)1 << 32);
}

bool mid_fwd_leads(int64_t M, int32_t N, int32_t K, int32_t E, int epilogue) {
    // K beyond 8192 (few experts, wide layers): tiles of twice the products per byte lead as soon as experts need two of the smaller
    // ones (8 experts of 176 rows, K = 28672: 470 against 516 us; K = 14336, 268 against 281; 320 rows 340 against 428)
    // - unless the experts' columns make at most 32 tiles, which leave most of the chip to K slices of 256 KB of sums a tile (4 experts of
    // H = 2048, K = 16384: 180 rows 155 -> 102 us, 258 rows 153 -> 117, 600 rows 250 -> 207; of H = 1024: 120 rows 114 -> 44, 400 rows
    // 104 -> 77; the worst of 72 pairs 7 % slower, 16 experts of H = 512, 400 rows).
    if (K > 8192 && M > (int64_t)112 * E && (int64_t)E * ((N + MR_BN - 1) / MR_BN) > 32) return false;
    int S;
    // without an epilogue of their own for GELU the 256 x 256 tiles leave it to a pass over two or three tensors
    const bool gelu = epilogue >= XMA_ROCM_EPI_GELU_TANH;
    const double pass = gelu ? ((epilogue & 1) ? 6.0 : 4.0) * M * N / 4.5e12 + 4e-6 : 0.;
    const int as = gelu ? XMA_ROCM_EPI_STORE : epilogue;
    // Even: as it was.  The model is one of launches of a few rounds; beyond them it flatters the smaller tiles, most where an epilogue
    // writes a second tensor, so what they have to be ahead by grows with the rounds.  5302 pairs of launches of random layers (2 to 128
    // experts, 97 to 8000 rows each), by epilogue, ms lost to choosing the smaller tiles where they were the slower ones, out of the ms
    // they won: SwiGLU 6.4 of 8.1 without this -> 0.5 of 7.3, GELU 7.0 of 10.0 -> 0.4 of 9.5, store 1.9 of 18.8 -> 1.3 of 18.5, SwiGLU
    // backward 1.4 of 15.0 -> 0.4 of 14.1; GELU backward 1.1 of 17.1 as it is.
    const double rounds = tiles_about(M, N, E, MR_BM) / MR_RUN;
    double even = 0.96;
    if (gelu && !(epilogue & 1))
        even -= rounds > 1 ? 0.15 * (rounds - 1) : 0.;
    else if (!gelu) {
        even -= rounds > 2.5 ? (epilogue == XMA_ROCM_EPI_SWIGLU ? 0.15 : 0.04) * (rounds - 2.5) : 0.;
        // Experts that need a second of the smaller tiles and fit into one of the larger, whose steps are shorter than 1.6 us then: its
        // waves skip the blocks without rows (0.79 of the predicted time at 96 to 160 rows, 0.9 beyond 256, from K = 3072 on).  25,500
        // pairs of random layers, 2 to 128 experts, 97 to 1400 rows each, ms lost and won by choosing the smaller tiles where they were the
        // slower and the faster ones: 20.3 and 377 without this -> 12.1 and 370 (64 experts of 125 rows, N = 2944, K = 6272: 484, 575 us).
        const double rows = (double)M / E, most = rows + 2.5 * sqrt(rows);
        if (K >= 3072 && most > MR_BM && most <= 256) even -= 0.08;
    }
    return mid_fwd_seconds(M, N, K, E, as, &S) < even * (tiles256_seconds(M, N, K, E, as) + pass);
}

int mid_fwd(const FwdArgs &a, int wt, int epi, int dtype, float *part, hipStream_t st) {
    if (dtype == XMA_ROCM_BF16) return wt ? mid_dispatch_fwd<__bf16, 1>(a, epi, part, st) : mid_dispatch_fwd<__bf16, 0>(a, epi, part, st);
    return wt ? mid_dispatch_fwd<_Float16, 1>(a, epi, part, st) : mid_dispatch_fwd<_Float16, 0>(a, epi, part, st);
}

bool mid_dw_leads(const DwArgs &a, int64_t M) {
    // From 40 rows per expert on in launches of two and more rounds of tiles (one and more where rows of dW start off 64-byte
    // boundaries), from 96 in smaller ones, whose time is the latency of a tile.  Small tiles / these, us: 5 experts of 688 x 256, 58 rows
    // each, 4.8 / 6.0; 20 of 1608 x 736, 72 rows, 1.5 rounds, 17.4 / 19.0; 89 of 600 x 832, 76 rows, 3.5 rounds, 34.5 / 25.5.
    const int64_t tiles = (int64_t)a.E * ((a.N_out + MR_BM - 1) / MR_BM) * ((a.K_in + MR_BN - 1) / MR_BN);
    return M > (tiles >= (mr_whole_lines(a) ? 2 : 1) * MR_RUN ? 40 : 96) * (int64_t)a.E;
}

bool mid_dw_takes(const DwArgs &a, int64_t M) {
    if (a.scale || (!a.dy_grouped && !a.x_grouped)) return false;
    const int64_t dy_rows = a.dy_grouped ? MR_K : (M + a.dy_fan_out - 1) / a.dy_fan_out, x_rows = a.x_grouped ? MR_K : (M + a.x_fan_out - 1) / a.x_fan_out;
    const int64_t tiles = (int64_t)a.E * ((a.N_out + MR_BM - 1) / MR_BM) * ((a.K_in + MR_BN - 1) / MR_BN);
    return M > 0 && M < ((int64_t)1 << 28) && tiles < ((int64_t)1 << 30) && dy_rows * a.lddy * 2 < ((int64_t)1 << 32) && x_rows * a.ldx * 2 < ((int64_t)1 << 32);
}

int mid_dw(const DwArgs &a, int dtype, hipStream_t st) {
    if (mr_whole_lines(a)) return dtype == XMA_ROCM_BF16 ? mid_dispatch_dw<__bf16, 1>(a, st) : mid_dispatch_dw<_Float16, 1>(a, st);
    return dtype == XMA_ROCM_BF16 ? mid_dispatch_dw<__bf16, 0>(a, st) : mid_dispatch_dw<_Float16, 0>(a, st);
}

} // namespace xma_rocm
