// The gate's share of the layer's backward, where nothing but the router weights hangs on the logits: a row of d_logits then has k
// values that are not zero, d_sel[t, j] at expert ids[t, j], and
//   d_gate[e] = sum over t, j with ids[t, j] = e of d_sel[t, j] x[t]          (E, H)
//   d_x[t]   += sum over j of d_sel[t, j] gate_weight[ids[t, j]]              (T, H)
// (the backward of gate(x), xma/layers/moe/__init__.py:182).  Two launches: gate_sums_kernel leaves fp32 sums of d_gate over ranges of
// the tokens, and the kernel that sums the k slots of the experts' d_x adds the second line and, in its first workgroups, the ranges.
//
// Measured against the stock products, the router's backward in a launch of its own and the product's addition to d_x in the last
// kernel (us; T tokens, H, E, k): 32768, 2048, 128, 8: 109 for the products -> 49 + 9 in the last kernel, whose gathered rows of the weight
// come from L2 beside the stream of the experts' rows; 16384, 2048, 64, 6: 61 -> 23; 8192, 4096, 8, 2: 80 -> 19; 1021, 2048, 8, 2: 24 -> 5;
// fp32, 512, 256, 8, 2: 21 -> 9, and one autograd node and three calls of torch less on the host: 288 -> 225 for forward and backward.
#include <type_traits>

#include "common.hpp"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int GT_THREADS = 256, GT_TOKENS = 64, GT_COLS = 128;
constexpr int GT_MAX_E = 128, GT_MAX_K = 32;
constexpr int GT_RUN = 512; // workgroups: two per compute unit

template <typename ET> struct Rows; // elements in memory, and 16 bytes of them
template <> struct Rows<__bf16> { typedef uint16_t type; };
template <> struct Rows<_Float16> { typedef uint16_t type; };
template <> struct Rows<float> { typedef float type; };

template <typename ET> __device__ __forceinline__ float to_float(typename Rows<ET>::type v) {
    if constexpr (sizeof(v) == 4)
        return v;
    else
        return Elem<ET>::lo((uint32_t)v);
}

// [64 rows][128 columns] of 16-bit elements as [64][16 chunks of 16 B], chunk c of row r at slot c ^ ((r & 3) << 2): byte offset
__device__ __forceinline__ int tile_at(int row, int col) { return row * 256 + (((col >> 3) ^ ((row & 3) << 2)) << 4) + (col & 7) * 2; }

// Byte offset of the fragment read of lane `lane` in the 32 columns from R0 on, k-rows 0 .. 15; those of rows 4 .. 7 (of each 8) lie 1024 behind
__device__ __forceinline__ int frag_at(int R0, int lane) {
    const int p = lane & 15, G = lane >> 4;
    return tile_at(((G >> 1) << 3) + (p >> 2), R0 + ((G & 1) << 4) + ((p & 3) << 2));
}
__device__ __forceinline__ u32x4 read_frag(const unsigned char *tile, int at) {
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4s *lds_v4s;
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(tile + at)));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(tile + at + 1024)));
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// sums[range][e][c] = sum over the range's tokens of d_logits[t][e] x[t][c], d_logits as a tile in LDS that holds d_sel at the selected
// experts and zeros elsewhere.  Workgroup = 128 columns x one range of tokens, 64 tokens a step; a wave owns 32 columns and all experts,
// EB blocks of 32 (v_mfma_f32_32x32x16 on 16-bit tiles through the transposing LDS read, v_mfma_f32_32x32x2_f32 on fp32, whose x needs
// no LDS).  KQ: slots of the 64 tokens per thread.  Reads x once per launch: bound by that stream, or by the two round trips of a range of
// one step.
template <typename ET, int EB, int KQ>
__global__ __launch_bounds__(GT_THREADS) void gate_sums_kernel(const typename Rows<ET>::type *__restrict__ x, int64_t ldx,
                                                               const typename Rows<ET>::type *__restrict__ d_sel,
                                                               const int32_t *__restrict__ ids, FastDiv k_div, int k, int64_t T, int H, int E,
                                                               int steps_per, float *__restrict__ sums) {
    typedef typename Rows<ET>::type T0;
    constexpr bool F32 = sizeof(T0) == 4;
    constexpr int PITCH = F32 ? EB * 32 * 4 : 256; // bytes of a row of the d_logits tile
    __shared__ __attribute__((aligned(16))) unsigned char s_d[GT_TOKENS * PITCH];
    __shared__ __attribute__((aligned(16))) unsigned char s_x[F32 ? 16 : GT_TOKENS * 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c0 = blockIdx.x * GT_COLS;
    const int64_t t_begin = (int64_t)blockIdx.y * steps_per * GT_TOKENS;
    const int64_t t_end = t_begin + (int64_t)steps_per * GT_TOKENS < T ? t_begin + (int64_t)steps_per * GT_TOKENS : T;
    for (int i = tid * 16; i < GT_TOKENS * PITCH; i += GT_THREADS * 16) *(u32x4 *)(s_d + i) = u32x4{0u, 0u, 0u, 0u};

    // this thread's parts of a step: slots tid + 256 q of the 64 k, and 16-bit chunks (row tid / 16 + 16 i, chunk tid % 16) or, fp32, the
    // 32 values (row 2 i + lane / 32, column lane % 32) of its wave
    int e_of[KQ];
    T0 d_of[KQ];
    u32x4 xr[F32 ? 1 : 4];
    float xf[F32 ? 32 : 1];
    auto fetch = [&](int64_t t0) {
        const int left = (int)(t_end - t0 < GT_TOKENS ? t_end - t0 : GT_TOKENS);
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            const int s = tid + GT_THREADS * q;
            e_of[q] = -1;
            if (s < left * k) {
                const int e = ids[t0 * k + s];
                e_of[q] = e < 0 ? 0 : (e >= E ? E - 1 : e); // never outside the tile
                d_of[q] = d_sel[t0 * k + s];
            }
        }
        if constexpr (F32) {
            const int c = c0 + 32 * wave + (lane & 31), r = lane >> 5;
#pragma unroll
            for (int i = 0; i < 32; ++i) xf[i] = 2 * i + r < left && c < H ? x[(t0 + 2 * i + r) * ldx + c] : 0.f;
        } else {
            const int c = c0 + (tid & 15) * 8, r = tid >> 4;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                xr[i] = 16 * i + r < left && c < H ? *(const u32x4 *)(x + (t0 + 16 * i + r) * ldx + c) : u32x4{0u, 0u, 0u, 0u};
        }
    };
    f32x16 acc[EB];
#pragma unroll
    for (int b = 0; b < EB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[b][v] = 0.f;
    if (t_begin < t_end) fetch(t_begin);
    for (int64_t t0 = t_begin; t0 < t_end; t0 += GT_TOKENS) {
        __syncthreads(); // the tiles of the step before have been read, its slots (or the first zeros) written
        int at[KQ];
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            at[q] = -1;
            if (e_of[q] >= 0) {
                const int row = (int)fastdiv((uint32_t)(tid + GT_THREADS * q), k_div);
                at[q] = F32 ? row * PITCH + e_of[q] * 4 : tile_at(row, e_of[q]);
                *(T0 *)(s_d + at[q]) = d_of[q];
            }
        }
        float xs[F32 ? 32 : 1];
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 32; ++i) xs[i] = xf[i];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) *(u32x4 *)(s_x + tile_at(16 * i + (tid >> 4), (tid & 15) * 8)) = xr[i];
        }
        __syncthreads();
        if (t0 + GT_TOKENS < t_end) fetch(t0 + GT_TOKENS);
        if constexpr (F32) {
#pragma unroll
            for (int i = 0; i < 32; ++i)
#pragma unroll
                for (int b = 0; b < EB; ++b) {
                    const float d = *(const float *)(s_d + (2 * i + (lane >> 5)) * PITCH + (32 * b + (lane & 31)) * 4);
                    acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(d, xs[i], acc[b], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const u32x4 p = read_frag(s_x + kk * 4096, frag_at(32 * wave, lane));
#pragma unroll
                for (int b = 0; b < EB; ++b) acc[b] = Elem<ET>::mfma(read_frag(s_d + kk * 4096, frag_at(32 * b, lane)), p, acc[b]);
            }
        }
        __syncthreads(); // read by all: its slots go back to zero
#pragma unroll
        for (int q = 0; q < KQ; ++q)
            if (at[q] >= 0) *(T0 *)(s_d + at[q]) = T0(0);
    }
    const int c = c0 + 32 * wave + (lane & 31);
    float *out = sums + (int64_t)blockIdx.y * E * H + c;
#pragma unroll
    for (int b = 0; b < EB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int e = 32 * b + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
            if (e < E && c < H) out[(int64_t)e * H] = acc[b][v];
        }
}

// d_x[t, c ..] = sum_j in[t k + j, c ..] (rounded; left out where `in` is NULL) + sum_j d_sel[t, j] gate_weight[ids[t, j], c ..] (rounded),
// a thread per 16 bytes; the first sum_blocks workgroups add the ranges of d_gate instead.
template <typename ET>
__global__ __launch_bounds__(GT_THREADS) void combine_gate_kernel(const typename Rows<ET>::type *__restrict__ in,
                                                                  const typename Rows<ET>::type *__restrict__ gate_weight,
                                                                  const typename Rows<ET>::type *__restrict__ d_sel,
                                                                  const int32_t *__restrict__ ids, typename Rows<ET>::type *__restrict__ d_x,
                                                                  int64_t T, int k, int H, int E, int chunks_per_row, FastDiv cpr_div,
                                                                  const float *__restrict__ sums, int ranges, int sum_blocks,
                                                                  typename Rows<ET>::type *__restrict__ d_gate) {
    typedef typename Rows<ET>::type T0;
    constexpr bool F32 = sizeof(T0) == 4;
    constexpr int V = 16 / sizeof(T0); // elements of a chunk
    if ((int)blockIdx.x < sum_blocks) {
        const int64_t i = ((int64_t)blockIdx.x * GT_THREADS + threadIdx.x) * 4, n = (int64_t)E * H; // n % 8 == 0
        if (i >= n) return;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
        for (int r = 0; r < ranges; ++r) s += *(const f32x4 *)(sums + r * n + i);
        if constexpr (F32)
            *(f32x4 *)(d_gate + i) = s;
        else
            *(u32x2 *)(d_gate + i) = u32x2{Elem<ET>::pack(s[0], s[1]), Elem<ET>::pack(s[2], s[3])};
        return;
    }
    const int64_t g = (int64_t)(blockIdx.x - sum_blocks) * GT_THREADS + threadIdx.x;
    if (g >= T * chunks_per_row) return;
    int64_t t;
    int c;
    split_row(g, chunks_per_row, cpr_div, t, c);
    c *= V;
    const T0 *row = in ? in + t * k * H + c : nullptr;
    float a[V], b[V];
#pragma unroll
    for (int v = 0; v < V; ++v) a[v] = b[v] = 0.f;
    auto add = [](float (&acc)[V], const u32x4 u, float s) {
        if constexpr (F32) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t bits = u[q];
                acc[q] += s * __builtin_bit_cast(float, bits);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                acc[2 * q] += s * Elem<ET>::lo(u[q]);
                acc[2 * q + 1] += s * Elem<ET>::hi(u[q]);
            }
        }
    };
    // N slots at a time: their experts, then the rows of either operand
    auto slots = [&](int j, auto N) {
        constexpr int n = decltype(N)::value;
        int e[n];
        float s[n];
        u32x4 u[n], w[n];
#pragma unroll
        for (int q = 0; q < n; ++q) e[q] = ids[t * k + j + q];
        if (row) {
#pragma unroll
            for (int q = 0; q < n; ++q) u[q] = __builtin_nontemporal_load((const u32x4 *)(row + (int64_t)(j + q) * H));
        }
#pragma unroll
        for (int q = 0; q < n; ++q) {
            e[q] = e[q] < 0 ? 0 : (e[q] >= E ? E - 1 : e[q]); // never outside the weight
            s[q] = to_float<ET>(d_sel[t * k + j + q]);
            w[q] = *(const u32x4 *)(gate_weight + (int64_t)e[q] * H + c);
        }
#pragma unroll
        for (int q = 0; q < n; ++q) {
            if (row) add(a, u[q], 1.f);
            add(b, w[q], s[q]);
        }
    };
    int j = 0;
    for (; j + 4 <= k; j += 4) slots(j, std::integral_constant<int, 4>());
    if (j + 2 <= k) slots(j, std::integral_constant<int, 2>()), j += 2;
    if (j < k) slots(j, std::integral_constant<int, 1>());
    u32x4 o;
    if constexpr (F32) {
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = __builtin_bit_cast(uint32_t, row ? a[q] + b[q] : b[q]);
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[q] = Elem<ET>::pack(b[2 * q], b[2 * q + 1]);
            if (row) {
                const uint32_t x = Elem<ET>::pack(a[2 * q], a[2 * q + 1]);
                o[q] = Elem<ET>::pack(Elem<ET>::lo(x) + Elem<ET>::lo(o[q]), Elem<ET>::hi(x) + Elem<ET>::hi(o[q]));
            }
        }
    }
    *(u32x4 *)(d_x + t * H + c) = o;
}

// Ranges of tokens: as many as make two workgroups per compute unit, of whole steps.
struct Ranges {
    int steps_per, count;
};
Ranges gate_ranges(int64_t T, int H) {
    const int64_t steps = (T + GT_TOKENS - 1) / GT_TOKENS, blocks = (H + GT_COLS - 1) / GT_COLS;
    const int64_t want = GT_RUN / blocks > 1 ? GT_RUN / blocks : 1, n = steps < want ? steps : want;
    const int64_t per = n ? (steps + n - 1) / n : 1;
    return {(int)per, (int)((steps + per - 1) / per)};
}

template <typename ET>
int gate_bwd(const void *x, int64_t ldx, const void *gate_weight, const void *d_sel, const int32_t *ids, const void *scattered, void *d_x,
             void *d_gate, int64_t T, int H, int E, int k, float *sums, hipStream_t st) {
    typedef typename Rows<ET>::type T0;
    const Ranges r = gate_ranges(T, H);
    if (d_gate) {
        const dim3 grid((H + GT_COLS - 1) / GT_COLS, r.count);
#define CALL(EB, KQ)                                                                                                                        \
    gate_sums_kernel<ET, EB, KQ><<<grid, GT_THREADS, 0, st>>>((const T0 *)x, ldx, (const T0 *)d_sel, ids, make_fastdiv((uint32_t)k), k, T, H, E, \
                                                              r.steps_per, sums)
#define CALL_EB(KQ) E <= 32 ? CALL(1, KQ) : E <= 64 ? CALL(2, KQ) : CALL(4, KQ)
        k <= 8 ? CALL_EB(2) : CALL_EB(8);
#undef CALL_EB
#undef CALL
        if (int rc = xma_check_launch("gate_sums_kernel")) return rc;
    }
    const int cpr = H * (int)sizeof(T0) / 16;
    const int64_t blocks = d_x ? (T * cpr + GT_THREADS - 1) / GT_THREADS : 0;
    XMA_REQUIRE(blocks < ((int64_t)1 << 30), XMA_ROCM_EUNSUPPORTED, "gate_bwd: too many rows");
    const int sum_blocks = d_gate ? (int)(((int64_t)E * H / 4 + GT_THREADS - 1) / GT_THREADS) : 0;
    combine_gate_kernel<ET><<<(unsigned)(blocks + sum_blocks), GT_THREADS, 0, st>>>(
        (const T0 *)scattered, (const T0 *)gate_weight, (const T0 *)d_sel, ids, (T0 *)d_x, T, k, H, E, cpr, make_fastdiv((uint32_t)cpr), sums,
        r.count, sum_blocks, (T0 *)d_gate);
    return xma_check_launch("combine_gate_kernel");
}

} // namespace

extern "C" int xma_rocm_gate_bwd_supported(int32_t H, int32_t E, int32_t k, int dtype) {
    return (dtype == XMA_ROCM_BF16 || dtype == XMA_ROCM_F16 || dtype == XMA_ROCM_F32) && H >= 8 && H % 8 == 0 && E >= 1 && E <= GT_MAX_E && k >= 1 &&
           k <= E && k <= GT_MAX_K;
}

extern "C" size_t xma_rocm_gate_bwd_workspace_bytes(int64_t T, int32_t H, int32_t E) {
    if (T <= 0 || H <= 0 || E <= 0) return 0;
    return (size_t)gate_ranges(T, H).count * (size_t)E * (size_t)H * sizeof(float);
}

int xma_gate_bwd_check(const char *what, const void *x, int64_t ldx, const void *gate_weight, const void *d_sel, const int32_t *ids,
                       const void *scattered, const void *d_x, const void *d_gate, int64_t T, int32_t H, int32_t E, int32_t k, int dtype,
                       const void *workspace, size_t workspace_bytes) {
    XMA_REQUIRE(xma_rocm_gate_bwd_supported(H, E, k, dtype), XMA_ROCM_EUNSUPPORTED, "%s: H=%d E=%d k=%d dtype=%d", what, H, E, k, dtype);
    const int es = dtype == XMA_ROCM_F32 ? 4 : 2;
    XMA_REQUIRE(T >= 1 && T * k < ((int64_t)1 << 31) && ldx >= H && ldx * es % 16 == 0, XMA_ROCM_EINVAL, "%s: T=%lld ldx=%lld", what,
                (long long)T, (long long)ldx);
    const uintptr_t all = (uintptr_t)x | (uintptr_t)gate_weight | (uintptr_t)scattered | (uintptr_t)d_x | (uintptr_t)d_gate | (uintptr_t)workspace;
    XMA_REQUIRE(d_sel && ids && (d_x || d_gate) && (!d_x || gate_weight) && (!d_gate || (x && workspace)) && (all & 15) == 0, XMA_ROCM_EINVAL,
                "%s: null or misaligned pointer", what);
    const size_t need = d_gate ? xma_rocm_gate_bwd_workspace_bytes(T, H, E) : 0;
    XMA_REQUIRE(workspace_bytes >= need, XMA_ROCM_EWORKSPACE, "%s: workspace of %zu bytes, %zu needed", what, workspace_bytes, need);
    return XMA_ROCM_OK;
}

int xma_gate_bwd(const void *x, int64_t ldx, const void *gate_weight, const void *d_sel, const int32_t *ids, const void *scattered, void *d_x,
                 void *d_gate, int64_t T, int32_t H, int32_t E, int32_t k, int dtype, void *workspace, size_t workspace_bytes, hipStream_t st) {
    if (int rc = xma_gate_bwd_check("gate_bwd", x, ldx, gate_weight, d_sel, ids, scattered, d_x, d_gate, T, H, E, k, dtype, workspace, workspace_bytes))
        return rc;
    float *sums = (float *)workspace;
    if (dtype == XMA_ROCM_BF16) return gate_bwd<__bf16>(x, ldx, gate_weight, d_sel, ids, scattered, d_x, d_gate, T, H, E, k, sums, st);
    if (dtype == XMA_ROCM_F16) return gate_bwd<_Float16>(x, ldx, gate_weight, d_sel, ids, scattered, d_x, d_gate, T, H, E, k, sums, st);
    return gate_bwd<float>(x, ldx, gate_weight, d_sel, ids, scattered, d_x, d_gate, T, H, E, k, sums, st);
}

extern "C" int xma_rocm_gate_bwd(const void *x, int64_t ldx, const void *gate_weight, const void *d_selected, const int32_t *ids, void *d_x,
                                 void *d_gate_weight, int64_t T, int32_t H, int32_t E, int32_t k, int dtype, void *workspace,
                                 size_t workspace_bytes, void *stream) {
    return xma_gate_bwd(x, ldx, gate_weight, d_selected, ids, nullptr, d_x, d_gate_weight, T, H, E, k, dtype, workspace, workspace_bytes,
                        (hipStream_t)stream);
}
