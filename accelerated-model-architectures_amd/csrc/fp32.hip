// fp32 variants of every op of the library (dtype XMA_ROCM_F32).
//
// The MoE layer is meant to run in bf16/fp16; fp32 is the dtype of parity runs against the CPU path and of the
// reference's own test grid.  These kernels are therefore written for exactness and simplicity, not for the roofline:
// v_mfma_f32_32x32x2_f32 with fp32 operands and accumulators (no reduced-precision pass anywhere), 64 x 64 or 128 x 128
// output tiles, operands staged through registers into k-major LDS tiles.  Schedule, operand roles, gather /
// scatter semantics and epilogues are those of the 16-bit kernels in grouped_gemm.hip:
//   forward / dX :  Q = activation rows (tokens),  P = weight rows (output features)
//   dW           :  Q = dY columns (out features), P = X columns (in features), K = tokens of the expert
// The MFMA "A" operand is the P fragment, so a lane owns output row (lane & 31) of a 32 x 32 block and four
// consecutive columns per accumulator quad.
#include "fp32.hpp"
#include "fp32_tiles.hpp"
#include "row_dot.hpp"

namespace {

constexpr int FTHREADS = 256;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Output tile of a workgroup: 64 TB x 64 TB, a quarter per wave (TB x TB blocks of 32 x 32).  A K step of the large tile
// is 2048 cycles of matrix pipe behind one step's loads.  The small one has 1024 and keeps the loads of two steps in
// flight: its launches have one or two workgroups per compute unit, so nothing else covers the latency.
template <int TB> struct Tile {
    static constexpr int DIM = 64 * TB, BK = f32_tile_step(64 * TB), SETS = 3 - TB;
    static constexpr int LD = DIM + 4; // floats per k-row of an LDS tile [BK][DIM + 4]: 16-byte aligned rows, conflict-free columns
    // K-contiguous source ([row][k]): 2 or 4 neighbouring threads share a row, two float4 per thread
    static __device__ __forceinline__ int row(int tid) { return TB == 2 ? tid >> 1 : tid >> 2; }
    static __device__ __forceinline__ int kc(int tid, int h) { return TB == 2 ? (tid & 1) * 8 + 4 * h : (tid & 3) * 4 + 16 * h; }
    // K-strided source ([k][row], rows contiguous): DIM / 4 neighbouring threads share a k
    static __device__ __forceinline__ int ks(int tid, int h) { return tid / (DIM / 4) + (BK / 2) * h; }
    static __device__ __forceinline__ int col(int tid) { return (tid % (DIM / 4)) * 4; }
};

struct TileRegs {
    f32x4 v[2];
};

// ---- operand tile loaders: DIM "rows" x BK k per tile, two float4 per thread
template <int TB> __device__ __forceinline__ void load_kcontig(TileRegs &r, const float *row_ptr, int k0, int K, int tid) {
    if (k0 + Tile<TB>::BK <= K) { // uniform: loads under a per-lane condition sit in branches of their own
#pragma unroll
        for (int h = 0; h < 2; ++h) r.v[h] = *(const f32x4 *)(row_ptr + k0 + Tile<TB>::kc(tid, h));
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = k0 + Tile<TB>::kc(tid, h);
        r.v[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (k < K) r.v[h] = *(const f32x4 *)(row_ptr + k); // K % 4 == 0: a float4 is inside or outside as a whole
    }
}
template <int TB> __device__ __forceinline__ void store_kcontig(float *tile, const TileRegs &r, int tid) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < 4; ++q) tile[(Tile<TB>::kc(tid, h) + q) * Tile<TB>::LD + Tile<TB>::row(tid)] = r.v[h][q];
}
template <int TB> __device__ __forceinline__ void store_kstrided(float *tile, const TileRegs &r, int tid) {
#pragma unroll
    for (int h = 0; h < 2; ++h) *(f32x4 *)(tile + Tile<TB>::ks(tid, h) * Tile<TB>::LD + Tile<TB>::col(tid)) = r.v[h];
}

template <int TB> __device__ __forceinline__ void zero_acc(f32x16 (&acc)[TB][TB]) {
#pragma unroll
    for (int j = 0; j < TB; ++j)
#pragma unroll
        for (int i = 0; i < TB; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][i][v] = 0.f;
}

// the BK k of the LDS tiles, MFMA steps of k = 2; the order of a sum over k does not depend on the tile
template <int TB>
__device__ __forceinline__ void mma_tiles(const float *sP, const float *sQ, f32x16 (&acc)[TB][TB], int wp, int wq, int lane) {
#pragma unroll
    for (int kk = 0; kk < Tile<TB>::BK / 2; ++kk) {
        const int k = 2 * kk + (lane >> 5);
        float p[TB], q[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            p[b] = sP[k * Tile<TB>::LD + wp + b * 32 + (lane & 31)];
            q[b] = sQ[k * Tile<TB>::LD + wq + b * 32 + (lane & 31)];
        }
#pragma unroll
        for (int j = 0; j < TB; ++j)
#pragma unroll
            for (int i = 0; i < TB; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(p[j], q[i], acc[j][i], 0, 0, 0);
    }
}

// The K loop.  LDS holds two steps, so a step has one barrier: the next one's operands go into the other place in front of this one's MFMAs,
// which cover them, and their registers are loaded again for the step after.  us, against two barriers and one place: x @ W^T of 16 experts of
// 250 rows, K = 2048, N = 1024 208 -> 184, 8 of 1000, K = 2048, N = 512 168 -> 150 (small tile); 8 of 2000, K = 2048, N = 512, dy @ W 303 ->
// 284 (large).
template <int TB, typename Load, typename Store, typename Multiply>
__device__ __forceinline__ void walk_k(int KT, Load load, Store store, Multiply multiply) {
    constexpr int SETS = Tile<TB>::SETS;
#pragma unroll
    for (int s = 0; s < SETS; ++s)
        if (s < KT) load(s, s);
    if (KT > 0) store(0, 0);
    if (SETS < KT) load(0, SETS);
    __syncthreads();
    for (int kt0 = 0; kt0 < KT; kt0 += SETS) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
            const int kt = kt0 + s;
            if (kt >= KT) break; // uniform
            if (kt + 1 < KT) {
                store((s + 1) % SETS, kt + 1); // everybody has read what was there before the last barrier
                if (kt + 1 + SETS < KT) load((s + 1) % SETS, kt + 1 + SETS);
            }
            multiply(kt);
            __syncthreads();
        }
    }
}

__device__ __forceinline__ float sigmoid_f32(float x) { return 1.0f / (1.0f + __expf(-x)); }

// ------------------------------------------------------------------------------------------------ forward / dX
template <int WT, int EPI, int TB>
__global__ __launch_bounds__(FTHREADS) void gemm_f32_kernel(const FwdArgs a) {
    typedef Tile<TB> T;
    extern __shared__ int s_pre[]; // [E + 1]
    __shared__ __attribute__((aligned(16))) float sQ[2][T::BK * T::LD];
    __shared__ __attribute__((aligned(16))) float sP[2][T::BK * T::LD];
    __shared__ int s_sched[2];
    const float *X = (const float *)a.X, *W = (const float *)a.W, *scale = (const float *)a.scale;
    float *out = (float *)a.out, *aux = (float *)a.aux;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int NT = (a.N + T::DIM - 1) / T::DIM;

    // expert-major schedule from the inclusive offsets: prefix sum of the experts' tiles by wave 0, 64 experts a step
    if (wave == 0) {
        int run = 0;
        for (int e0 = 0; e0 < a.E; e0 += WAVE) {
            const int e = e0 + lane;
            int tiles = 0;
            if (e < a.E) tiles = (int)((a.offs[e] - (e ? a.offs[e - 1] : 0) + T::DIM - 1) / T::DIM) * NT;
            int incl = tiles;
#pragma unroll
            for (int d = 1; d < WAVE; d <<= 1) {
                const int t = __shfl_up(incl, d);
                if (lane >= d) incl += t;
            }
            if (e < a.E) s_pre[e] = run + incl - tiles;
            run += __shfl(incl, WAVE - 1);
        }
        if (lane == 0) {
            s_pre[a.E] = run;
            s_sched[0] = -1;
        }
    }
    __syncthreads();
    const int L = blockIdx.x;
    for (int e = tid; e < a.E; e += FTHREADS)
        if (s_pre[e] <= L && L < s_pre[e + 1]) {
            s_sched[0] = e;
            s_sched[1] = L - s_pre[e];
        }
    __syncthreads();
    const int e = s_sched[0];
    if (e < 0) return; // the grid is an upper bound
    const int64_t row_lo = e ? a.offs[e - 1] : 0, row_hi = a.offs[e];
    const int tiles_m = (int)((row_hi - row_lo + T::DIM - 1) / T::DIM);
    const int64_t row0 = row_lo + (int64_t)(s_sched[1] % tiles_m) * T::DIM;
    const int n0 = (s_sched[1] / tiles_m) * T::DIM;
    const int rows_valid = (int)((row_hi - row0 < T::DIM) ? row_hi - row0 : T::DIM);

    // loader set-up
    const float *q_row; // this thread's activation row (K-contiguous source)
    {
        int r = T::row(tid);
        if (r >= rows_valid) r = rows_valid - 1; // duplicates, masked at the store
        const int64_t n = row0 + r;
        const int64_t src = a.x_grouped ? n : (int64_t)fastdiv((uint32_t)a.idx[n], a.fan_div);
        q_row = X + src * a.ldx;
    }
    const float *We = W + (int64_t)e * a.w_es;
    const float *p_row = nullptr; // WT == 0: this thread's weight row
    int p_col = 0;                // WT == 1: first of this thread's 4 columns
    if (WT == 0) {
        int r = n0 + T::row(tid);
        if (r >= a.N) r = a.N - 1;
        p_row = We + (int64_t)r * a.ldw;
    } else {
        p_col = n0 + T::col(tid);
        if (p_col >= a.N) p_col = a.N - 4; // masked at the store
    }
    auto load_p = [&](TileRegs &r, int k0) {
        if (WT == 0) {
            load_kcontig<TB>(r, p_row, k0, a.K, tid);
        } else if (k0 + T::BK <= a.K) { // uniform
#pragma unroll
            for (int h = 0; h < 2; ++h) r.v[h] = *(const f32x4 *)(We + (int64_t)(k0 + T::ks(tid, h)) * a.ldw + p_col);
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = k0 + T::ks(tid, h);
                r.v[h] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (k < a.K) r.v[h] = *(const f32x4 *)(We + (int64_t)k * a.ldw + p_col);
            }
        }
    };

    f32x16 acc[TB][TB];
    zero_acc<TB>(acc);
    const int wq = (wave & 1) * 32 * TB, wp = (wave >> 1) * 32 * TB;
    if (a.bias) { // the expert's bias is the first term of every sum (see the epilogue for a lane's columns)
        const float *b = (const float *)a.bias + (int64_t)e * a.bias_es;
#pragma unroll
        for (int j = 0; j < TB; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                int col = n0 + wp + j * 32 + g * 8 + (lane >> 5) * 4;
                if (col > a.N - 4) col = a.N - 4;
                const f32x4 v = *(const f32x4 *)(b + col);
#pragma unroll
                for (int i = 0; i < TB; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[j][i][4 * g + q] = v[q];
            }
    }
    const int KT = (a.K + T::BK - 1) / T::BK;
    TileRegs rq[T::SETS], rp[T::SETS]; // the next SETS steps
    auto load = [&](int s, int kt) {
        load_kcontig<TB>(rq[s], q_row, kt * T::BK, a.K, tid); // zeros past K
        load_p(rp[s], kt * T::BK);
    };
    auto store = [&](int s, int kt) {
        store_kcontig<TB>(sQ[kt & 1], rq[s], tid);
        if (WT == 0)
            store_kcontig<TB>(sP[kt & 1], rp[s], tid);
        else
            store_kstrided<TB>(sP[kt & 1], rp[s], tid);
    };
    walk_k<TB>(KT, load, store, [&](int kt) { mma_tiles<TB>(sP[kt & 1], sQ[kt & 1], acc, wp, wq, lane); });

    // epilogue: lane owns row (lane & 31) of each 32-row block, 4 consecutive columns per quad
    const int lrow = lane & 31, lhalf = lane >> 5;
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        const int r = wq + i * 32 + lrow;
        if (r >= rows_valid) continue;
        const int64_t n = row0 + r;
        int64_t sidx = 0;
        if (!a.y_grouped || scale) sidx = a.idx[n];
        const int64_t dst = a.y_grouped ? n : sidx;
        const float sc = scale ? scale[sidx] : 1.f;
#pragma unroll
        for (int j = 0; j < TB; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int col = n0 + wp + j * 32 + g * 8 + lhalf * 4;
                if (col >= a.N) continue;
                const f32x4 v = {acc[j][i][4 * g] * sc, acc[j][i][4 * g + 1] * sc, acc[j][i][4 * g + 2] * sc,
                                 acc[j][i][4 * g + 3] * sc};
                if (EPI == XMA_ROCM_EPI_STORE) {
                    *(f32x4 *)(out + dst * a.ldo + col) = v;
                } else if (EPI == XMA_ROCM_EPI_SWIGLU) {
                    if (out) *(f32x4 *)(out + dst * a.ldo + col) = v;
                    // columns are (gate, up, gate, up)
                    float2 h = {v[1] * v[0] * sigmoid_f32(v[0]), v[3] * v[2] * sigmoid_f32(v[2])};
                    *(float2 *)(aux + dst * a.ldaux + (col >> 1)) = h;
                } else { // SWIGLU_BWD: v = d h of 4 columns; z and dz have 8 columns (g, u) x 4, grouped rows
                    const f32x4 z0 = *(const f32x4 *)(aux + n * a.ldaux + 2 * col);
                    const f32x4 z1 = *(const f32x4 *)(aux + n * a.ldaux + 2 * col + 4);
                    const float zz[8] = {z0[0], z0[1], z0[2], z0[3], z1[0], z1[1], z1[2], z1[3]};
                    float o[8];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float gg = zz[2 * q], uu = zz[2 * q + 1];
                        const float sg = sigmoid_f32(gg), silu = gg * sg;
                        o[2 * q] = v[q] * uu * (sg + silu * (1.f - sg));
                        o[2 * q + 1] = v[q] * silu;
                    }
                    *(f32x4 *)(out + n * a.ldo + 2 * col) = f32x4{o[0], o[1], o[2], o[3]};
                    *(f32x4 *)(out + n * a.ldo + 2 * col + 4) = f32x4{o[4], o[5], o[6], o[7]};
                }
            }
    }
}

// ------------------------------------------------------------------------------------------------ dW
template <int TB> __global__ __launch_bounds__(FTHREADS) void dw_f32_kernel(const DwArgs a) {
    typedef Tile<TB> T;
    __shared__ __attribute__((aligned(16))) float sQ[2][T::BK * T::LD];
    __shared__ __attribute__((aligned(16))) float sP[2][T::BK * T::LD];
    const float *DY = (const float *)a.DY, *X = (const float *)a.X, *scale = (const float *)a.scale;
    float *DW = (float *)a.DW;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int OT = (a.N_out + T::DIM - 1) / T::DIM, IT = (a.K_in + T::DIM - 1) / T::DIM;
    const int e = blockIdx.x / (OT * IT), rem = blockIdx.x % (OT * IT);
    const int o0 = (rem / IT) * T::DIM, i0 = (rem % IT) * T::DIM;
    const int64_t row_lo = e ? a.offs[e - 1] : 0, row_hi = a.offs[e];
    const int rows = (int)(row_hi - row_lo);
    const int KT = (rows + T::BK - 1) / T::BK;
    int q_col = o0 + T::col(tid), p_col = i0 + T::col(tid);
    if (q_col >= a.N_out) q_col = a.N_out - 4; // masked at the store
    if (p_col >= a.K_in) p_col = a.K_in - 4;

    // k-rows are tokens of the expert: a thread takes two rows of a step, through the index if the operand is in scattered order; dY may
    // carry a per-token scale.  The indices of a step are fetched with the operands of the one before it in the same registers, so that
    // no load waits for another in front of the MFMAs.
    const bool gathers = !a.dy_grouped || !a.x_grouped || scale;
    TileRegs rq[T::SETS], rp[T::SETS];
    uint32_t idx[T::SETS][2];
    float scales[T::SETS][2];
    auto load_idx = [&](int s, int kt) {
        if (!gathers) return; // uniform
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = kt * T::BK + T::ks(tid, h);
            idx[s][h] = (uint32_t)a.idx[row_lo + (k < rows ? k : rows - 1)];
        }
    };
    auto load = [&](int s, int kt) {
        if (kt == s) load_idx(s, kt); // of the first step in these registers; uniform
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = kt * T::BK + T::ks(tid, h), at = k < rows ? k : rows - 1; // past the last row: zeros, below
            const int64_t n = row_lo + at;
            const int64_t dsrc = a.dy_grouped ? n : (int64_t)fastdiv(idx[s][h], a.dy_div);
            const int64_t xsrc = a.x_grouped ? n : (int64_t)fastdiv(idx[s][h], a.x_div);
            rq[s].v[h] = *(const f32x4 *)(DY + dsrc * a.lddy + q_col);
            rp[s].v[h] = *(const f32x4 *)(X + xsrc * a.ldx + p_col);
            if (scale) scales[s][h] = scale[idx[s][h]];
        }
        if (kt + T::SETS < KT) load_idx(s, kt + T::SETS);
    };
    auto store = [&](int s, int kt) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (scale) rq[s].v[h] *= scales[s][h];
            if (kt * T::BK + T::BK > rows && kt * T::BK + T::ks(tid, h) >= rows) rq[s].v[h] = rp[s].v[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        store_kstrided<TB>(sQ[kt & 1], rq[s], tid);
        store_kstrided<TB>(sP[kt & 1], rp[s], tid);
    };

    f32x16 acc[TB][TB];
    zero_acc<TB>(acc);
    const int wq = (wave & 1) * 32 * TB, wp = (wave >> 1) * 32 * TB;
    walk_k<TB>(KT, load, store, [&](int kt) { mma_tiles<TB>(sP[kt & 1], sQ[kt & 1], acc, wp, wq, lane); });
    // every element of DW[e] is written, zeros for an expert without tokens
    const int lrow = lane & 31, lhalf = lane >> 5;
    float *DWe = DW + (int64_t)e * a.dw_es;
#pragma unroll
    for (int i = 0; i < TB; ++i) {
        const int o = o0 + wq + i * 32 + lrow;
        if (o >= a.N_out) continue;
#pragma unroll
        for (int j = 0; j < TB; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int col = i0 + wp + j * 32 + g * 8 + lhalf * 4;
                if (col >= a.K_in) continue;
                *(f32x4 *)(DWe + (int64_t)o * a.lddw + col) =
                    f32x4{acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]};
            }
    }
}

// ------------------------------------------------------------------------------------------------ elementwise
// one thread per float4 of the output
__global__ __launch_bounds__(FTHREADS) void combine_f32_kernel(const float *in, int64_t ld_in, const float *w, float *y,
                                                                int64_t ldy, int64_t T, int k, int cpr, const float *addend, int64_t ld_add) {
    const int64_t id = (int64_t)blockIdx.x * FTHREADS + threadIdx.x;
    if (id >= T * cpr) return;
    const int64_t t = id / cpr;
    const int c = (int)(id % cpr) * 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
        const float s = w ? w[t * k + j] : 1.f;
        acc += s * *(const f32x4 *)(in + (t * k + j) * ld_in + c);
    }
    if (addend) acc += *(const f32x4 *)(addend + t * ld_add + c);
    *(f32x4 *)(y + t * ldy + c) = acc;
}

// one wave per (token, slot): d_w[t, j] = <in[t k + j, :], dy[t, :]>
__global__ __launch_bounds__(FTHREADS) void combine_bwd_f32_kernel(const float *in, int64_t ld_in, const float *dy,
                                                                    int64_t lddy, float *d_w, int64_t rows, int k, int H) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * (FTHREADS / 64) + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int64_t t = row / k;
    const float acc = row_dot<float>(in + row * ld_in, dy + t * lddy, H, lane);
    if (lane == 0) d_w[row] = acc;
}

__global__ __launch_bounds__(FTHREADS) void group_f32_kernel(const float *A, int64_t lda, const int64_t *idx, float *out,
                                                              int64_t ldo, const float *coeff, int64_t M, int cpr,
                                                              int fan_out) {
    const int64_t id = (int64_t)blockIdx.x * FTHREADS + threadIdx.x;
    if (id >= M * cpr) return;
    const int64_t n = id / cpr;
    const int c = (int)(id % cpr) * 4;
    const int64_t s = idx[n];
    f32x4 v = *(const f32x4 *)(A + (s / fan_out) * lda + c);
    if (coeff) v *= coeff[s];
    *(f32x4 *)(out + n * ldo + c) = v;
}

// y[r, c] = up * gate * sigmoid(gate), x = (gate, up) interleaved; one thread per 4 outputs
__global__ __launch_bounds__(FTHREADS) void swiglu_fwd_f32_kernel(const float *x, int64_t ldx, float *y, int64_t ldy,
                                                                   int64_t rows, int cpr) {
    const int64_t id = (int64_t)blockIdx.x * FTHREADS + threadIdx.x;
    if (id >= rows * cpr) return;
    const int64_t r = id / cpr;
    const int c = (int)(id % cpr) * 4;
    const f32x4 a = *(const f32x4 *)(x + r * ldx + 2 * c), b = *(const f32x4 *)(x + r * ldx + 2 * c + 4);
    *(f32x4 *)(y + r * ldy + c) = f32x4{a[1] * a[0] * sigmoid_f32(a[0]), a[3] * a[2] * sigmoid_f32(a[2]),
                                        b[1] * b[0] * sigmoid_f32(b[0]), b[3] * b[2] * sigmoid_f32(b[2])};
}

__global__ __launch_bounds__(FTHREADS) void swiglu_bwd_f32_kernel(const float *x, int64_t ldx, const float *dy, int64_t lddy,
                                                                   float *dx, int64_t lddx, int64_t rows, int cpr) {
    const int64_t id = (int64_t)blockIdx.x * FTHREADS + threadIdx.x;
    if (id >= rows * cpr) return;
    const int64_t r = id / cpr;
    const int c = (int)(id % cpr) * 4;
    const f32x4 d = *(const f32x4 *)(dy + r * lddy + c);
    const f32x4 a = *(const f32x4 *)(x + r * ldx + 2 * c), b = *(const f32x4 *)(x + r * ldx + 2 * c + 4);
    const float zz[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    float o[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float gg = zz[2 * q], uu = zz[2 * q + 1];
        const float sg = sigmoid_f32(gg), silu = gg * sg;
        o[2 * q] = d[q] * uu * (sg + silu * (1.f - sg));
        o[2 * q + 1] = d[q] * silu;
    }
    *(f32x4 *)(dx + r * lddx + 2 * c) = f32x4{o[0], o[1], o[2], o[3]};
    *(f32x4 *)(dx + r * lddx + 2 * c + 4) = f32x4{o[4], o[5], o[6], o[7]};
}

inline int blocks_for(int64_t work) { return (int)((work + FTHREADS - 1) / FTHREADS); }

// The table of the experts' tiles is behind the operands' two steps, 34.8 KB: together they pass 64 KB from 7678 experts on.
constexpr int F32_MAX_E = 8192, F32_TABLE_BYTES = (F32_MAX_E + 1) * (int)sizeof(int);
template <int WT, int TB> int launch_gemm(const FwdArgs &a, int epi, int grid, hipStream_t st) {
    auto run = [&](auto kernel) {
        if (int rc = xma_set_max_lds_once((const void *)kernel, F32_TABLE_BYTES)) return rc;
        kernel<<<grid, FTHREADS, (size_t)(a.E + 1) * sizeof(int), st>>>(a);
        return xma_check_launch("gemm_f32_kernel");
    };
    if (epi == XMA_ROCM_EPI_STORE) return run(gemm_f32_kernel<WT, XMA_ROCM_EPI_STORE, TB>);
    if (epi == XMA_ROCM_EPI_SWIGLU) return run(gemm_f32_kernel<WT, XMA_ROCM_EPI_SWIGLU, TB>);
    return run(gemm_f32_kernel<WT, XMA_ROCM_EPI_SWIGLU_BWD, TB>);
}

} // namespace

int f32_scatter2scatter(const FwdArgs &a, int w_is_kn, int epilogue, hipStream_t st) {
    const bool small = f32_small_tile(a.M, a.N, a.K, a.E);
    const int dim = small ? 64 : 128;
    const int64_t grid = (a.M / dim + a.E) * ((a.N + dim - 1) / dim); // sum_e ceil(c_e / dim) <= floor(M / dim) + E
    XMA_REQUIRE(grid < ((int64_t)1 << 31), XMA_ROCM_EUNSUPPORTED, "scatter2scatter (fp32): grid too large");
    XMA_REQUIRE(a.E <= F32_MAX_E, XMA_ROCM_EUNSUPPORTED, "scatter2scatter (fp32): E=%d > %d", a.E, F32_MAX_E);
    if (small) return w_is_kn ? launch_gemm<1, 1>(a, epilogue, (int)grid, st) : launch_gemm<0, 1>(a, epilogue, (int)grid, st);
    return w_is_kn ? launch_gemm<1, 2>(a, epilogue, (int)grid, st) : launch_gemm<0, 2>(a, epilogue, (int)grid, st);
}

int f32_group_bwd_W(const DwArgs &a, int64_t M, hipStream_t st) {
    const bool small = f32_small_tile_dw(M, a.N_out, a.K_in, a.E);
    const int64_t grid = a.E * f32_tiles(a.N_out, a.K_in, small ? 64 : 128);
    XMA_REQUIRE(grid < ((int64_t)1 << 31), XMA_ROCM_EUNSUPPORTED, "group_bwd_W (fp32): grid too large");
    if (small)
        dw_f32_kernel<1><<<(int)grid, FTHREADS, 0, st>>>(a);
    else
        dw_f32_kernel<2><<<(int)grid, FTHREADS, 0, st>>>(a);
    return xma_check_launch("dw_f32_kernel");
}

int f32_combine(const void *in, int64_t ld_in, const void *w, const void *addend, int64_t ld_add, void *y, int64_t ldy, int64_t T, int k, int H, hipStream_t st) {
    const int cpr = H / 4;
    combine_f32_kernel<<<blocks_for(T * cpr), FTHREADS, 0, st>>>((const float *)in, ld_in, (const float *)w, (float *)y, ldy,
                                                                 T, k, cpr, (const float *)addend, ld_add);
    return xma_check_launch("combine_f32_kernel");
}

int f32_combine_bwd(const void *in, int64_t ld_in, const void *dy, int64_t lddy, void *d_w, int64_t T, int k, int H,
                    hipStream_t st) {
    const int64_t rows = T * k;
    const int64_t blocks = (rows + (FTHREADS / 64) - 1) / (FTHREADS / 64);
    combine_bwd_f32_kernel<<<(int)blocks, FTHREADS, 0, st>>>((const float *)in, ld_in, (const float *)dy, lddy, (float *)d_w,
                                                             rows, k, H);
    return xma_check_launch("combine_bwd_f32_kernel");
}

int f32_group(const void *A, int64_t lda, const int64_t *idx, void *out, int64_t ldo, const void *coeff, int64_t M, int K,
              int fan_out, hipStream_t st) {
    const int cpr = K / 4;
    group_f32_kernel<<<blocks_for(M * cpr), FTHREADS, 0, st>>>((const float *)A, lda, idx, (float *)out, ldo,
                                                               (const float *)coeff, M, cpr, fan_out);
    return xma_check_launch("group_f32_kernel");
}

int f32_swiglu_packed_forward(const void *x, int64_t ldx, void *y, int64_t ldy, int64_t rows, int cols_out, hipStream_t st) {
    const int cpr = cols_out / 4;
    swiglu_fwd_f32_kernel<<<blocks_for(rows * cpr), FTHREADS, 0, st>>>((const float *)x, ldx, (float *)y, ldy, rows, cpr);
    return xma_check_launch("swiglu_fwd_f32_kernel");
}

int f32_swiglu_packed_backward(const void *x, int64_t ldx, const void *dy, int64_t lddy, void *dx, int64_t lddx, int64_t rows,
                               int cols_out, hipStream_t st) {
    const int cpr = cols_out / 4;
    swiglu_bwd_f32_kernel<<<blocks_for(rows * cpr), FTHREADS, 0, st>>>((const float *)x, ldx, (const float *)dy, lddy,
                                                                       (float *)dx, lddx, rows, cpr);
    return xma_check_launch("swiglu_bwd_f32_kernel");
}
