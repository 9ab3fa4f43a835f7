// Gradient of the experts' bias: per-expert column sums of a row-major matrix whose rows are taken in grouped order
// (optionally through the scattered index, optionally times a per-row scale).  HBM-bound: every row is read once.
#include "common.hpp"

namespace {

constexpr int CS_COLS = 128;                   // columns per workgroup: a wave reads 256 (fp32: 512) contiguous bytes of a row
constexpr int CS_UNROLL = 4;                   // rows a wave has in flight

template <typename T> struct Pair; // two neighbouring elements of a row as floats
template <> struct Pair<float> {
    static __device__ __forceinline__ float2 load(const void *row, int c) { return *(const float2 *)((const float *)row + c); }
    static __device__ __forceinline__ float scalar(const void *v, int64_t i) { return ((const float *)v)[i]; }
    static __device__ __forceinline__ void store(void *row, int c, float a, float b) { *(float2 *)((float *)row + c) = make_float2(a, b); }
};
template <> struct Pair<__bf16> {
    static __device__ __forceinline__ float2 load(const void *row, int c) {
        const uint32_t w = *(const uint32_t *)((const uint16_t *)row + c);
        return make_float2(Elem<__bf16>::lo(w), Elem<__bf16>::hi(w));
    }
    static __device__ __forceinline__ float scalar(const void *v, int64_t i) { return Elem<__bf16>::lo(((const uint16_t *)v)[i]); }
    static __device__ __forceinline__ void store(void *row, int c, float a, float b) {
        *(uint32_t *)((uint16_t *)row + c) = Elem<__bf16>::pack(a, b);
    }
};
template <> struct Pair<_Float16> {
    static __device__ __forceinline__ float2 load(const void *row, int c) {
        const uint32_t w = *(const uint32_t *)((const uint16_t *)row + c);
        return make_float2(Elem<_Float16>::lo(w), Elem<_Float16>::hi(w));
    }
    static __device__ __forceinline__ float scalar(const void *v, int64_t i) { return Elem<_Float16>::lo(((const uint16_t *)v)[i]); }
    static __device__ __forceinline__ void store(void *row, int c, float a, float b) {
        *(uint32_t *)((uint16_t *)row + c) = Elem<_Float16>::pack(a, b);
    }
};

// out[e, c] = sum over the grouped rows n of expert e of A[src(n), c] * scale[idx[n]], src(n) = n (idx == NULL) or
// idx[n] / fan_out.  Workgroup (column block, expert); the rows are dealt to the waves round-robin and added in a
// fixed order (per wave in row order, then the waves in order), so the result does not depend on timing.  Experts
// without rows get zeros.
// A workgroup walks its expert's rows in steps of one round trip to memory each.  Launches of few workgroups are bound by
// these, so they get 16 waves with 4 rows in flight, 64 rows a step (measured against 4 waves with 4 rows: 16 experts of 300
// rows, 1024 / 4096 columns 11.3 -> 4.5 / 22.9 -> 8.8 us; of 4096 rows, 4096 columns 384 -> 127).  From four workgroups per CU
// on, 4 waves each fill the chip, and the larger workgroups only wait for their own last waves (2048 workgroups of 16 / 300
// rows: 3.0 / 26.4 us with 4 waves, 5.7 / 28.3 with 16; of 1024 rows 126 / 129).  With up to 16 rows per expert, one step or
// less, the larger workgroups cost 0.1 to 0.3 us of 2 to 2.4; the host does not know the number of rows.  8 rows in flight
// instead of 4 are slower on both sides (16 waves, 512 workgroups of 4096 rows 140 against 127 us; 4 waves, 2048 workgroups
// of 1024 rows 139 against 126).
constexpr int CS_FEW_BLOCKS = 1024;
template <typename T, int CS_PHASES>
__global__ __launch_bounds__(CS_PHASES * WAVE) void expert_column_sums_kernel(const void *__restrict__ A, int64_t lda,
                                                                        const int64_t *__restrict__ idx, FastDiv fan_div,
                                                                        const void *__restrict__ scale,
                                                                        const int64_t *__restrict__ offs, void *__restrict__ out,
                                                                        int64_t ldo, int N) {
    __shared__ float2 s_part[CS_PHASES][WAVE];
    constexpr int ES = sizeof(T);
    const int e = blockIdx.y, lane = threadIdx.x & 63, phase = threadIdx.x >> 6;
    int c = blockIdx.x * CS_COLS + 2 * lane;
    const bool col_ok = c < N;
    if (!col_ok) c = N - 2; // clamped, never stored
    const int64_t lo = e ? offs[e - 1] : 0, hi = offs[e];
    float s0 = 0.f, s1 = 0.f;
    for (int64_t r0 = lo + phase; r0 < hi; r0 += CS_UNROLL * CS_PHASES) {
        float2 v[CS_UNROLL];
        float w[CS_UNROLL];
#pragma unroll
        for (int u = 0; u < CS_UNROLL; ++u) {
            const int64_t r = r0 + u * CS_PHASES;
            v[u] = make_float2(0.f, 0.f);
            w[u] = 1.f;
            if (r < hi) {
                int64_t src = r;
                if (idx) {
                    const int64_t s = idx[r];
                    src = fastdiv((uint32_t)s, fan_div);
                    if (scale) w[u] = Pair<T>::scalar(scale, s);
                }
                v[u] = Pair<T>::load((const char *)A + src * lda * ES, c);
            }
        }
#pragma unroll
        for (int u = 0; u < CS_UNROLL; ++u) s0 += v[u].x * w[u], s1 += v[u].y * w[u];
    }
    s_part[phase][lane] = make_float2(s0, s1);
    __syncthreads();
    if (phase == 0 && col_ok) {
        float a = 0.f, b = 0.f;
#pragma unroll
        for (int p = 0; p < CS_PHASES; ++p) a += s_part[p][lane].x, b += s_part[p][lane].y;
        Pair<T>::store((char *)out + (int64_t)e * ldo * ES, c, a, b);
    }
}

// The same where rows are whole 16-byte pieces: a lane takes one (V columns), so a load of a wave covers 64 V / 128 rows of the
// workgroup's 128 columns instead of one, and a step of 16 waves 256 rows of 16-bit elements instead of 64.  The rows of a wave meet by
// lane exchanges, then the waves that have rows as above: a fixed order as well.  us, a piece of 4 bytes per lane / these, bf16, grouped
// rows and rows gathered and scaled: 16 experts of 512 rows, 1024 columns 6.6 / 4.2, 13.2 / 6.2; 64 of 1500, 2048 columns 158 / 68 (5.8
// TB/s), 278 / 78; 128 of 2048, 1536 columns 237 / 140, 563 / 167; 8 of 8 rows, 1024 columns 2.4 / 2.7, 2.6 / 2.8, where nothing is to be gained.
template <typename T, int CS_PHASES>
__global__ __launch_bounds__(CS_PHASES * WAVE) void expert_column_sums_wide_kernel(const void *__restrict__ A, int64_t lda,
                                                                             const int64_t *__restrict__ idx, FastDiv fan_div,
                                                                             const void *__restrict__ scale,
                                                                             const int64_t *__restrict__ offs, void *__restrict__ out,
                                                                             int64_t ldo, int N) {
    constexpr int ES = sizeof(T), V = 16 / ES, LANES = CS_COLS / V, ROWS = WAVE / LANES;
    __shared__ __attribute__((aligned(16))) float s_part[CS_PHASES][CS_COLS];
    const int e = blockIdx.y, lane = threadIdx.x & 63, phase = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int c = blockIdx.x * CS_COLS + V * (lane % LANES);
    if (c >= N) c = N - V; // never stored
    const int64_t lo = e ? offs[e - 1] : 0, hi = offs[e];
    float sum[V];
#pragma unroll
    for (int q = 0; q < V; ++q) sum[q] = 0.f;
    for (int64_t r0 = lo + phase * ROWS + lane / LANES; r0 < hi; r0 += CS_UNROLL * CS_PHASES * ROWS) {
        u32x4 v[CS_UNROLL];
        float w[CS_UNROLL];
#pragma unroll
        for (int u = 0; u < CS_UNROLL; ++u) {
            const int64_t r = r0 + u * (CS_PHASES * ROWS);
            v[u] = u32x4{0u, 0u, 0u, 0u};
            w[u] = 0.f;
            if (r < hi) {
                int64_t src = r;
                w[u] = 1.f;
                if (idx) {
                    const int64_t s = idx[r];
                    src = fastdiv((uint32_t)s, fan_div);
                    if (scale) w[u] = Pair<T>::scalar(scale, s);
                }
                v[u] = *(const u32x4 *)((const char *)A + (src * lda + c) * ES);
            }
        }
#pragma unroll
        for (int u = 0; u < CS_UNROLL; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (ES == 4) {
                    const uint32_t bits = v[u][q];
                    sum[q] += __builtin_bit_cast(float, bits) * w[u];
                } else {
                    sum[2 * q] += Elem<T>::lo(v[u][q]) * w[u];
                    sum[2 * q + 1] += Elem<T>::hi(v[u][q]) * w[u];
                }
            }
    }
    const int64_t full = (hi - lo + ROWS - 1) / ROWS;
    const int waves = __builtin_amdgcn_readfirstlane((int)(full < CS_PHASES ? full : CS_PHASES)); // that have rows
    if (phase < waves) {
#pragma unroll
        for (int d = LANES; d < WAVE; d <<= 1)
#pragma unroll
            for (int q = 0; q < V; ++q) sum[q] += __shfl_xor(sum[q], d);
        if (lane < LANES) {
#pragma unroll
            for (int q = 0; q < V; q += 4) *(float4 *)&s_part[phase][V * lane + q] = make_float4(sum[q], sum[q + 1], sum[q + 2], sum[q + 3]);
        }
    }
    __syncthreads();
    const int col = 2 * lane;
    if (phase == 0 && (int)blockIdx.x * CS_COLS + col < N) {
        float a = 0.f, b = 0.f;
        for (int p = 0; p < waves; ++p) a += s_part[p][col], b += s_part[p][col + 1];
        Pair<T>::store((char *)out + (int64_t)e * ldo * ES, blockIdx.x * CS_COLS + col, a, b);
    }
}

} // namespace

extern "C" int xma_rocm_expert_column_sums(const void *A, int64_t lda, const int64_t *sorted_scattered_idxs, int32_t fan_out,
                                           const void *row_scale, const int64_t *expert_offsets, void *out, int64_t ldo,
                                           int32_t N, int32_t E, int dtype, void *stream) {
    XMA_REQUIRE(dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16 || dtype == XMA_ROCM_F32, XMA_ROCM_EUNSUPPORTED,
                "expert_column_sums: dtype %d", dtype);
    XMA_REQUIRE(N >= 2 && N % 2 == 0 && E >= 1 && E <= 65535 && fan_out >= 1 && lda % 2 == 0 && ldo % 2 == 0 && lda >= N && ldo >= N,
                XMA_ROCM_EINVAL, "expert_column_sums: N=%d E=%d fan_out=%d lda=%lld ldo=%lld (N and the leading dimensions even)", N,
                E, fan_out, (long long)lda, (long long)ldo);
    XMA_REQUIRE(A && expert_offsets && out && ((uintptr_t)A & 7) == 0 && ((uintptr_t)out & 7) == 0, XMA_ROCM_EINVAL,
                "expert_column_sums: null or misaligned pointer");
    XMA_REQUIRE(!row_scale || sorted_scattered_idxs, XMA_ROCM_EINVAL,
                "expert_column_sums: the row scale is indexed through sorted_scattered_idxs");
    const dim3 grid((N + CS_COLS - 1) / CS_COLS, E);
    hipStream_t st = (hipStream_t)stream;
    const FastDiv fd = make_fastdiv((uint32_t)fan_out);
    const int v = dtype == XMA_ROCM_F32 ? 4 : 8; // elements of a 16-byte piece
    const bool wide = N % v == 0 && lda % v == 0 && ((uintptr_t)A & 15) == 0;
#define CS_LAUNCH(T, PHASES)                                                                                       \
    (wide ? expert_column_sums_wide_kernel<T, PHASES> : expert_column_sums_kernel<T, PHASES>)<<<grid, PHASES * WAVE, 0, st>>>( \
        A, lda, sorted_scattered_idxs, fd, row_scale, expert_offsets, out, ldo, N)
#define CS_LAUNCH_T(T) few ? CS_LAUNCH(T, 16) : CS_LAUNCH(T, 4)
    const bool few = (int64_t)grid.x * grid.y < CS_FEW_BLOCKS;
    if (dtype == XMA_ROCM_BF16)
        CS_LAUNCH_T(__bf16);
    else if (dtype == XMA_ROCM_F16)
        CS_LAUNCH_T(_Float16);
    else
        CS_LAUNCH_T(float);
#undef CS_LAUNCH_T
#undef CS_LAUNCH
    return xma_check_launch("expert_column_sums_kernel");
}
