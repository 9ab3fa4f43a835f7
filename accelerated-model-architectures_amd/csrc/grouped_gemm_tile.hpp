// Pieces that the grouped GEMM kernels of 256-row and of 128-row tiles share: compile-time loops, LDS-DMA loads through a buffer
// descriptor, and the epilogues of a tile (plain store with optional row scale and scatter, SwiGLU forward and backward).
#pragma once

#include "gemm_common.hpp"

namespace xma_rocm {

typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int N> struct IC {
    static constexpr int value = N;
};
// compile-time loop: f(IC<0>{}), ..., f(IC<N-1>{}) - the index is a constant expression inside f (asm immediates)
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(IC<N - 1>{});
    }
}

__device__ __forceinline__ uint32_t lds_addr_of(const void *p) {
    return (uint32_t)(size_t)((__attribute__((address_space(3))) const char *)p);
}

// Epilogue staging in LDS, private to a wave: one 32-row block of its 128 x 128 corner as 16-bit values (rows padded
// by 16 bytes against bank conflicts), followed by the 32 x 64 block of SwiGLU activations.
constexpr int EPI_Z_STRIDE = 128 * 2 + 16, EPI_H_STRIDE = 64 * 2 + 16;
// Internal epilogue code beside the public XMA_ROCM_EPI_*: SWIGLU_BWD with the second output FwdArgs::aux2.  A variant of
// its own, so that the launches without that output keep their code and register allocation unchanged.
constexpr int EPI_SWIGLU_BWD_SCALED_ACT = 3;
// And both of them with the gradient of the row scale, FwdArgs::dots (256-row tiles).  Compiled into the launches that do not ask for it, its
// arithmetic made them 1.00 - 1.03 times as long as the kernel ahead of it, without it they are 0.95 - 1.00 (262144 rows of H = 2048, I = 768
// 897 -> 904 us with it, 911 -> 893 without, in turn on two boxes; 24000 of H = 512, I = 1032 68.8 -> 69.8, 70.0 -> 66.2).
constexpr int EPI_SWIGLU_BWD_DOTS = 8, EPI_SWIGLU_BWD_SCALED_ACT_DOTS = 9;
__host__ __device__ constexpr bool epi_dots(int epi) { return epi == EPI_SWIGLU_BWD_DOTS || epi == EPI_SWIGLU_BWD_SCALED_ACT_DOTS; }
__host__ __device__ constexpr bool epi_scaled_act(int epi) { return epi == EPI_SWIGLU_BWD_SCALED_ACT || epi == EPI_SWIGLU_BWD_SCALED_ACT_DOTS; }
__host__ __device__ constexpr bool epi_swiglu_bwd(int epi) { return epi == XMA_ROCM_EPI_SWIGLU_BWD || epi_scaled_act(epi) || epi_dots(epi); }
// z and h = gelu(z), both (M, N); dz = gelu'(z) d h: FwdArgs::erf_form says which GELU
constexpr int EPI_GELU = XMA_ROCM_EPI_GELU_TANH, EPI_GELU_BWD = XMA_ROCM_EPI_GELU_TANH_BWD;
constexpr int EPI_WAVE_BYTES = 32 * EPI_Z_STRIDE + 32 * EPI_H_STRIDE;
// SwiGLU backward stages 32 rows of 256 pre-activation columns per wave
constexpr int EPI_BWD_STRIDE = 256 * 2 + 16, EPI_BWD_WAVE_BYTES = 32 * EPI_BWD_STRIDE;

// LDS written by some lanes of a wave is read by others of the same wave: instructions of one wave reach the LDS in
// order, so only the compiler has to be kept from reordering.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T> __device__ __forceinline__ uint32_t one_bits();
template <> __device__ __forceinline__ uint32_t one_bits<__bf16>() { return 0x3f80u; }
template <> __device__ __forceinline__ uint32_t one_bits<_Float16>() { return 0x3c00u; }

// Buffer loads: uniform 48-bit base, 32-bit byte offset per lane.  An offset at or past the size in the descriptor
// (BUF_OUTSIDE) reads zeros.
constexpr uint32_t BUF_OUTSIDE = 0xffffffffu;
__device__ __forceinline__ i32x4 buf_desc(const void *base, uint32_t bytes = 0xfffffff0u) {
    // the base is uniform by construction; where the register allocation keeps it in vector registers all the same, the two
    // readfirstlane bring it back (they fold away where it already is scalar)
    const uint64_t b = (uint64_t)base;
    i32x4 d;
    d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    d[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32) & 0xffff);
    d[2] = __builtin_amdgcn_readfirstlane((int)bytes);
    d[3] = 0x00020000;       // raw 32-bit data
    return d;
}
// a * b + c in two 32-bit instructions (the compiler's 64-bit multiply-add would take a register pair for the result)
__device__ __forceinline__ uint32_t mul_add_u32(uint32_t a, uint32_t b, uint32_t c) {
    uint32_t m = a * b;
    asm("" : "+v"(m));
    return m + c;
}
__device__ __forceinline__ void lds_dma16_buf(i32x4 desc, uint32_t off, uint32_t lds_base, uint32_t stage) {
    asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds" ::"s"(lds_base), "s"(stage), "v"(off),
                 "s"(desc)
                 : "memory", "m0", "scc");
}

// Scattered index and row scale of a lane's row in each of the (up to four) 32-row blocks of its wave (row wq + 32 i + lane % 32
// of the tile, clamped to the last valid row), when the caller has fetched them ahead of the epilogue.
struct EpiRows {
    int idx[4];
    float sc[4];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_buffer(const void *p, uint32_t bytes) {
    const uint64_t base = (uint64_t)p, lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base);
    const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(base >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(lo | hi << 32), 0, __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}
// The rows of a tile in one of its grouped matrices: 16-byte accesses at row, by 32-bit offsets from the tile's first row.  What lies past
// the last valid row is outside the buffer: loads read zeros and stores are dropped, so no row is clamped, and an address is one addition
// where 64-bit ones take a clamp and a product each, a fifth of the instructions of the SwiGLU backward's epilogue.  On its own that
// gives those launches nothing (the epilogue's vector ALU is busy for 0.6 of it either way); it makes room for `dots`.
struct RowBuffer {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t lane_off, ld_bytes;
    __device__ __forceinline__ RowBuffer(const uint16_t *m, int64_t ld, int64_t row0, int rows_valid, int lane_row, int col) {
        ld_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(2 * ld));
        rsrc = uniform_buffer(m + row0 * ld, (uint32_t)rows_valid * ld_bytes);
        lane_off = mul_add_u32((uint32_t)lane_row, ld_bytes, (uint32_t)col * 2);
    }
    __device__ __forceinline__ u32x4 load(int row) const {
        return __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_off + (uint32_t)row * ld_bytes, 0, 0);
    }
    __device__ __forceinline__ void store(int row, u32x4 v) const {
        __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, lane_off + (uint32_t)row * ld_bytes, 0, 0);
    }
};

// Whether the offsets of a launch's epilogue fit: 256 rows of every grouped matrix in 2^32 - 1 bytes, the scattered one in 2^32 pieces of 16.
inline bool row_offsets_fit(const FwdArgs &a) {
    const int64_t most = ((int64_t)1 << 23) - 1;
    return (a.y_grouped ? a.ldo <= most : a.M * (a.ldo / 8) < ((int64_t)1 << 32)) && (!a.aux || a.ldaux <= most) && (!a.aux2 || a.ldaux2 <= most);
}

// ---- epilogue of one tile of 64 NI rows x 256 columns (2 x 2 waves of NI 32-row blocks x 128 columns); smem: staging area that no
// wave reads operand tiles from any more
// FIT: the launch's offsets fit (row_offsets_fit).
template <typename T, int EPI, int NI = 4, int FIT = 0>
__device__ __forceinline__ void tile_epilogue(const FwdArgs &a, f32x16 (&acc)[4][NI], unsigned char *smem, int64_t row0,
                                              int rows_valid, int n0, int tid, int only_i = -1,
                                              const EpiRows *pre = nullptr) {
    // only_i >= 0: just the 32-row block only_i of every wave (the fix-up kernel spreads a tile over four workgroups)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wq = (wave & 1) * (32 * NI), wp = (wave >> 1) * 128; // wave's corner inside the tile
    // lane owns row (lane & 31) of each 32-row block; quad g of tile (j, i) holds
    //      columns n0 + wp + 32 j + 8 g + 4 (lane >> 5) + {0..3}
    const int lrow = lane & 31, lhalf = lane >> 5;
    if constexpr (EPI == EPI_GELU_BWD) {
        // as the SwiGLU backward below, with z and dz as wide as d h: 32 rows of 128 columns come in and leave through the
        // staging area of the plain store
        if (__builtin_amdgcn_readfirstlane(n0 + wp) >= a.N) return; // this wave's columns all lie past N
        unsigned char *stage = smem + wave * EPI_WAVE_BYTES;
        const int piece = (n0 + wp + (lane & 15) * 8 < a.N) ? (lane & 15) : 0;
        const int cz = n0 + wp + piece * 8;
        // a copy per form: a branch per element keeps the elements' instructions apart (16 experts of 512 rows, K = 1024, N = 4096: 128
        // against 112 us here, 128 against 107 in the forward; plain store 87, and a pass over the tensors 33 and 39)
        auto blocks = [&](auto ERF) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int rbase = wq + i * 32;
            if (rbase >= rows_valid) break; // wave-uniform
            u32x4 zin[8];
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                int r = rbase + 4 * it + (lane >> 4);
                if (r >= rows_valid) r = rows_valid - 1;
                zin[it] = *(const u32x4 *)(a.aux + (row0 + r) * a.ldaux + cz);
            }
            int r_lane = rbase + lrow;
            if (r_lane >= rows_valid) r_lane = rows_valid - 1;
            float sc = 1.f;
            if (a.scale) sc = pre ? pre->sc[i] : Elem<T>::lo((uint32_t)a.scale[a.idx[row0 + r_lane]]);
#pragma unroll
            for (int it = 0; it < 8; ++it) *(u32x4 *)(stage + (4 * it + (lane >> 4)) * EPI_Z_STRIDE + (lane & 15) * 16) = zin[it];
            wave_lds_sync();
            unsigned char *mine = stage + lrow * EPI_Z_STRIDE + lhalf * 8;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    u32x2 *zp = (u32x2 *)(mine + (j * 32 + g * 8) * 2);
                    const u32x2 z = *zp;
                    float d[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        d[q] = acc[j][i][4 * g + q] * sc * gelu_grad((q & 1) ? Elem<T>::hi(z[q >> 1]) : Elem<T>::lo(z[q >> 1]), ERF.value, sigmoidf_fast);
                    *zp = u32x2{Elem<T>::pack(d[0], d[1]), Elem<T>::pack(d[2], d[3])};
                }
            wave_lds_sync();
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                int br = 4 * it + (lane >> 4);
                if (rbase + br >= rows_valid) br = rows_valid - 1 - rbase;
                *(u32x4 *)(a.out + (row0 + rbase + br) * a.ldo + cz) = *(const u32x4 *)(stage + br * EPI_Z_STRIDE + piece * 16);
            }
            wave_lds_sync(); // the next block overwrites the area
        }
        };
        if (a.erf_form)
            blocks(IC<1>{});
        else
            blocks(IC<0>{});
    } else if constexpr (!epi_swiglu_bwd(EPI)) {
        // A store instruction of the accumulator layout would touch 32 rows with 16 bytes each.  Instead every
        // 32-row block goes through a wave-private LDS area and leaves as whole rows: 16 lanes x 16 bytes per row of
        // 128 columns (8 lanes per row of the 64 activation columns), i.e. full 128-byte lines.
        // Stores are unconditional: a lane whose row or column lies outside the tile's valid part repeats the store of a
        // lane inside it (same address, same data, read from the same place of the staging area).  Under a per-lane
        // condition every store sits in a branch of its own, with its addresses spilled and reloaded around it.
        if (__builtin_amdgcn_readfirstlane(n0 + wp) >= a.N) return; // this wave's columns all lie past N
        unsigned char *stage = smem + wave * EPI_WAVE_BYTES;
        unsigned char *z_w = stage + lrow * EPI_Z_STRIDE + lhalf * 8;
        unsigned char *h_w = stage + 32 * EPI_Z_STRIDE + lrow * EPI_H_STRIDE + lhalf * 4;
        const int z_piece = (n0 + wp + (lane & 15) * 8 < a.N) ? (lane & 15) : 0; // this lane's 8 output columns on the way out
        const int h_piece = (n0 + wp + (lane & 7) * 16 < a.N) ? (lane & 7) : 0;  // and its 8 activation columns
        const int cz = n0 + wp + z_piece * 8, ch = ((n0 + wp) >> 1) + h_piece * 8;
        const bool write_z = (EPI == XMA_ROCM_EPI_STORE) || a.out != nullptr;
        // scattered row and scale of this lane's row in each of the blocks, fetched before the first store:
        // loads and stores retire in order, so a load between the blocks would wait for the stores before it
        int idx_i[4] = {0, 0, 0, 0};
        float sc_i[4] = {1.f, 1.f, 1.f, 1.f};
        if (!a.y_grouped || a.scale != nullptr) {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                int r = wq + i * 32 + lrow;
                if (r >= rows_valid) r = rows_valid - 1; // duplicates are computed and stored again
                idx_i[i] = pre ? pre->idx[i] : (int)a.idx[row0 + r];
            }
        }
        if (a.scale) {
#pragma unroll
            for (int i = 0; i < NI; ++i) sc_i[i] = pre ? pre->sc[i] : Elem<T>::lo((uint32_t)a.scale[idx_i[i]]);
        }
        // copies of the loop: without a row scale the 256 multiplications by one are left out; rows in grouped order
        // need no exchange of row indices between lanes
        auto blocks = [&](auto SCALED, auto GROUPED) {
        const int last = rows_valid - 1;
        constexpr bool buf = FIT && GROUPED.value, units = FIT && !GROUPED.value;
        const RowBuffer out_b(a.out, a.ldo, buf ? row0 : 0, buf && write_z ? rows_valid : 0, wq + (lane >> 4), cz);
        const RowBuffer aux_b(a.aux, a.ldaux, buf ? row0 : 0, buf ? rows_valid : 0, wq + (lane >> 3), ch);
        uint16_t *out0 = a.out + (GROUPED.value ? row0 * a.ldo : 0) + cz;
        uint16_t *aux0 = a.aux + (GROUPED.value ? row0 * a.ldaux : 0) + ch;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int rbase = wq + i * 32;
            if (rbase >= rows_valid) break; // wave-uniform
            if (only_i >= 0 && i != only_i) continue;
            const float sc = sc_i[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float v0 = acc[j][i][4 * g], v1 = acc[j][i][4 * g + 1];
                    float v2 = acc[j][i][4 * g + 2], v3 = acc[j][i][4 * g + 3];
                    if constexpr (SCALED.value) v0 *= sc, v1 *= sc, v2 *= sc, v3 *= sc;
                    const uint32_t z0 = Elem<T>::pack(v0, v1), z1 = Elem<T>::pack(v2, v3);
                    u32x2 o = {z0, z1};
                    *(u32x2 *)(z_w + (j * 32 + g * 8) * 2) = o;
                    if constexpr (EPI == XMA_ROCM_EPI_SWIGLU) {
                        // columns are (gate, up, gate, up); the activation is taken from the rounded
                        // pre-activations, exactly what a separate pass over the stored z would see
                        const float g0 = Elem<T>::lo(z0), u0 = Elem<T>::hi(z0);
                        const float g1 = Elem<T>::lo(z1), u1 = Elem<T>::hi(z1);
                        const float h0 = u0 * g0 * sigmoidf_fast(g0), h1 = u1 * g1 * sigmoidf_fast(g1);
                        *(uint32_t *)(h_w + (j * 16 + g * 4) * 2) = Elem<T>::pack(h0, h1);
                    }
                }
            }
            wave_lds_sync();
            if constexpr (units) {
                // rows past the last valid one hold its sums and its place again, as everywhere here
                const uint32_t place = (uint32_t)idx_i[i] * (uint32_t)(a.ldo >> 3);
                if (write_z) {
#pragma unroll
                    for (int it = 0; it < 8; ++it) {
                        const u32x4 v = *(const u32x4 *)(stage + (4 * it + (lane >> 4)) * EPI_Z_STRIDE + z_piece * 16);
                        *(u32x4 *)(out0 + (int64_t)(uint32_t)__shfl((int)place, 4 * it + (lane >> 4)) * 8) = v;
                    }
                }
            } else if (write_z) {
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    if constexpr (buf) {
                        out_b.store(i * 32 + 4 * it, *(const u32x4 *)(stage + (4 * it + (lane >> 4)) * EPI_Z_STRIDE + z_piece * 16));
                        continue;
                    }
                    int r = rbase + 4 * it + (lane >> 4);
                    if (r > last) r = last;
                    const u32x4 v = *(const u32x4 *)(stage + (r - rbase) * EPI_Z_STRIDE + z_piece * 16);
                    const int64_t d = GROUPED.value ? r : __shfl(idx_i[i], r - rbase);
                    *(u32x4 *)(out0 + d * a.ldo) = v;
                }
            }
            if constexpr (EPI == EPI_GELU) { // the activations of the rounded z take the same way out
                wave_lds_sync();
                auto activate = [&](auto ERF) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            u32x2 *zp = (u32x2 *)(z_w + (j * 32 + g * 8) * 2);
                            const u32x2 z = *zp;
                            float h[4];
#pragma unroll
                            for (int q = 0; q < 4; ++q) h[q] = gelu((q & 1) ? Elem<T>::hi(z[q >> 1]) : Elem<T>::lo(z[q >> 1]), ERF.value, sigmoidf_fast);
                            *zp = u32x2{Elem<T>::pack(h[0], h[1]), Elem<T>::pack(h[2], h[3])};
                        }
                };
                if (a.erf_form)
                    activate(IC<1>{});
                else
                    activate(IC<0>{});
                wave_lds_sync();
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    int r = rbase + 4 * it + (lane >> 4);
                    if (r > last) r = last;
                    const u32x4 v = *(const u32x4 *)(stage + (r - rbase) * EPI_Z_STRIDE + z_piece * 16);
                    *(u32x4 *)(a.aux + (row0 + r) * a.ldaux + cz) = v;
                }
            }
            if constexpr (EPI == XMA_ROCM_EPI_SWIGLU) {
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    if constexpr (buf) {
                        aux_b.store(i * 32 + 8 * it, *(const u32x4 *)(stage + 32 * EPI_Z_STRIDE + (8 * it + (lane >> 3)) * EPI_H_STRIDE + h_piece * 16));
                        continue;
                    }
                    int r = rbase + 8 * it + (lane >> 3);
                    if (r > last) r = last;
                    const u32x4 v = *(const u32x4 *)(stage + 32 * EPI_Z_STRIDE + (r - rbase) * EPI_H_STRIDE + h_piece * 16);
                    const int64_t d = GROUPED.value ? r : __shfl(idx_i[i], r - rbase);
                    *(u32x4 *)(aux0 + d * a.ldaux) = v;
                }
            }
            wave_lds_sync(); // the next block overwrites the area
        }
        };
        if constexpr (EPI == EPI_GELU) { // grouped rows, no scale
            blocks(IC<0>{}, IC<1>{});
        } else if constexpr (EPI == XMA_ROCM_EPI_SWIGLU) { // the layer's form: grouped rows, no scale
            if (a.y_grouped && !a.scale)
                blocks(IC<0>{}, IC<1>{});
            else if (a.y_grouped)
                blocks(IC<1>{}, IC<1>{});
            else
                blocks(IC<1>{}, IC<0>{});
        } else {
            if (a.scale) {
                if (a.y_grouped) blocks(IC<1>{}, IC<1>{}); else blocks(IC<1>{}, IC<0>{});
            } else {
                if (a.y_grouped) blocks(IC<0>{}, IC<1>{}); else blocks(IC<0>{}, IC<0>{});
            }
        }
    } else {
        // SwiGLU backward: the accumulators are d h for the wave's 128 columns; z and dz have twice as many (gate, up
        // interleaved).  Each 32-row block of z comes in as whole rows (2 rows of 512 bytes per instruction) through
        // the wave-private LDS area, every lane turns its own 16-byte pieces into dz in place, and the block leaves
        // the same way.  The z rows of block i + 1 are requested before the stores of block i go out: loads and
        // stores retire in order, so a load issued behind the stores would wait for them.
        unsigned char *stage = smem + wave * EPI_BWD_WAVE_BYTES;
        unsigned char *row_io = stage + (lane >> 5) * EPI_BWD_STRIDE + (lane & 31) * 16; // + 2 it rows (way in)
        unsigned char *mine = stage + lrow * EPI_BWD_STRIDE + lhalf * 16;                // + (32 j + 8 g) * 4 bytes
        // Loads and stores of this epilogue are unconditional: a lane whose column lies outside the tile's valid part, and without FIT one
        // whose row does, repeats the access of a lane inside it (same address, and for stores the same data, read from the same place
        // of the staging area); with FIT a row outside lies outside the buffer.  Memory operations under a per-lane condition sit in branches, and the compiler then waits
        // for all of them (vmcnt(0)) where it would otherwise count: every block would wait for the stores of the one
        // before it to complete before it could bring its own rows of z into LDS.
        // this wave's 128 columns lie past N: nothing to do, and nothing in here joins other waves (the value is uniform;
        // readfirstlane tells the compiler so, which keeps the branch scalar)
        if (__builtin_amdgcn_readfirstlane(n0 + wp) >= a.N) return;
        const int piece = (2 * (n0 + wp) + (lane & 31) * 8 < 2 * a.N) ? (lane & 31) : 0; // piece 0 is inside N
        const int cz = 2 * (n0 + wp) + piece * 8; // this lane's 8 columns of z / dz on the way in and out
        float sc_i[4];
        // The gradient of a row's scale (the router weight) is <d h, h>: a lane owns a row here and has both at hand, so it costs one
        // multiply-add per value, an exchange between the row's two lanes and 4 bytes per row and wave.  A pass over the expert outputs
        // that forms it as <dy, expert_out> reads k T H of them again.  Forward + backward, 262144 rows of H = 2048, I = 768: 7861 -> 7695 us;
        // 98304 of I = 1408: 5547 -> 5510; 16384 of H = 4096, I = 14336: equal.
        constexpr bool dots = epi_dots(EPI);
        static_assert(!dots || NI == 4, "the 256-row tiles only");
        const int cols = a.N - (n0 + wp); // columns from here on are not the wave's: what they hold is dropped
        // no condition on these stores either: for the rows past the last valid one they lie outside the buffer
        const __amdgpu_buffer_rsrc_t dots_b = uniform_buffer(a.dots, dots ? a.dots_bytes : 0u);
        int idx_i[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            int r = wq + i * 32 + lrow;
            if (r >= rows_valid) r = rows_valid - 1;
            sc_i[i] = 1.f;
            if (a.scale) sc_i[i] = pre ? pre->sc[i] : Elem<T>::lo((uint32_t)a.scale[a.idx[row0 + r]]);
            if (dots) idx_i[i] = pre ? pre->idx[i] : (int)a.idx[row0 + r];
        }
        const RowBuffer z_b(a.aux, a.ldaux, FIT ? row0 : 0, FIT ? rows_valid : 0, wq + (lane >> 5), cz);
        const RowBuffer dz_b(a.out, a.ldo, FIT ? row0 : 0, FIT ? rows_valid : 0, wq + (lane >> 5), cz);
        u32x4 zin[16];
        auto load_block = [&](int i) {
#pragma unroll
            for (int it = 0; it < 16; ++it) {
                if constexpr (FIT) {
                    zin[it] = z_b.load(i * 32 + 2 * it);
                    continue;
                }
                int r = wq + i * 32 + 2 * it + (lane >> 5);
                if (r >= rows_valid) r = rows_valid - 1;
                zin[it] = *(const u32x4 *)(a.aux + (row0 + r) * a.ldaux + cz);
            }
        };
        const int i_first = only_i >= 0 ? only_i : 0, i_last = only_i >= 0 ? only_i : NI - 1;
        if (wq + i_first * 32 < rows_valid) load_block(i_first);
        // HS: a second output, the activations scaled by the row scale, (M, N) in grouped order.  A lane keeps its 128
        // values of a block, packed in 32 registers, until the dz rows have left; then the block takes the same way out
        // through the staging area (32 rows of 128 columns, the layout of the plain store epilogue).  With four blocks the 32
        // registers are accumulation registers - the 64 of the block's own accumulators are free by then - written and read
        // with v_accvgpr moves: as ordinary variables they push the kernel's register allocation into spilling.  (Storing
        // each quad straight from registers, 8 bytes per lane = 16 bytes of 32 rows per instruction, measured slower.)
        auto park = [](uint32_t v) {
            if constexpr (NI < 4) return v;
            uint32_t r;
            asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(r) : "v"(v));
            return r;
        };
        auto unpark = [](uint32_t r) {
            if constexpr (NI < 4) return r;
            uint32_t v;
            asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(r));
            return v;
        };
        auto blocks = [&](auto HS) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (wq + i * 32 >= rows_valid) break; // wave-uniform
            if (i < i_first || i > i_last) continue;
            // with two waves per SIMD the other one covers the latency, and the 64 registers are wanted for the next tile
            if (NI < 4 && i > i_first) load_block(i);
#pragma unroll
            for (int it = 0; it < 16; ++it) *(u32x4 *)(row_io + 2 * it * EPI_BWD_STRIDE) = zin[it];
            if (NI == 4 && i < i_last && wq + (i + 1) * 32 < rows_valid) load_block(i + 1);
            wave_lds_sync();
            const float sc = sc_i[i];
            uint32_t hs[HS.value ? 32 : 1];
            float dot = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    u32x4 *zp = (u32x4 *)(mine + (j * 32 + g * 8) * 4);
                    const u32x4 z = *zp;
                    u32x4 o;
                    float hv[4], dq = 0.f;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float dh = acc[j][i][4 * g + q] * sc;
                        const float gg = Elem<T>::lo(z[q]), uu = Elem<T>::hi(z[q]);
                        const float sg = sigmoidf_fast(gg), silu = gg * sg;
                        o[q] = Elem<T>::pack(dh * uu * (sg + silu * (1.f - sg)), dh * silu);
                        hv[q] = uu * silu * sc;
                        if constexpr (dots) dq += acc[j][i][4 * g + q] * (uu * silu);
                    }
                    if constexpr (dots) dot += (j * 32 + g * 8 < cols) ? dq : 0.f; // uniform: N is a multiple of 8
                    *zp = o;
                    if constexpr (HS.value != 0) {
                        hs[2 * (j * 4 + g)] = park(Elem<T>::pack(hv[0], hv[1]));
                        hs[2 * (j * 4 + g) + 1] = park(Elem<T>::pack(hv[2], hv[3]));
                    }
                }
            }
            wave_lds_sync();
#pragma unroll
            for (int it = 0; it < 16; ++it) {
                if constexpr (FIT) {
                    dz_b.store(i * 32 + 2 * it, *(const u32x4 *)(stage + (2 * it + (lane >> 5)) * EPI_BWD_STRIDE + piece * 16));
                    continue;
                }
                int br = 2 * it + (lane >> 5); // row of the block; the block's first row is valid
                if (wq + i * 32 + br >= rows_valid) br = rows_valid - 1 - (wq + i * 32);
                const u32x4 v = *(const u32x4 *)(stage + br * EPI_BWD_STRIDE + piece * 16);
                *(u32x4 *)(a.out + (row0 + wq + i * 32 + br) * a.ldo + cz) = v;
            }
            if constexpr (dots) {
                dot += __shfl_xor(dot, 32);
                const uint32_t at = mul_add_u32((uint32_t)idx_i[i], a.dots_ld, (uint32_t)(n0 + wp) >> 7) * 4;
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, dot), dots_b, wq + i * 32 + lrow < rows_valid ? at : BUF_OUTSIDE, 0, 0);
            }
            wave_lds_sync(); // the next block overwrites the area
            if constexpr (HS.value != 0) {
                unsigned char *h_w = stage + lrow * EPI_Z_STRIDE + lhalf * 8;
                const int hpiece = (n0 + wp + (lane & 15) * 8 < a.N) ? (lane & 15) : 0; // as above: no store is conditional
                const int ch = n0 + wp + hpiece * 8; // this lane's 8 activation columns on the way out
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *(u32x2 *)(h_w + (j * 32 + g * 8) * 2) = u32x2{unpark(hs[2 * (j * 4 + g)]), unpark(hs[2 * (j * 4 + g) + 1])};
                wave_lds_sync();
                const RowBuffer h_b(a.aux2, a.ldaux2, FIT ? row0 : 0, FIT ? rows_valid : 0, wq + (lane >> 4), ch);
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    if constexpr (FIT) {
                        h_b.store(i * 32 + 4 * it, *(const u32x4 *)(stage + (4 * it + (lane >> 4)) * EPI_Z_STRIDE + hpiece * 16));
                        continue;
                    }
                    int br = 4 * it + (lane >> 4);
                    if (wq + i * 32 + br >= rows_valid) br = rows_valid - 1 - (wq + i * 32);
                    const u32x4 v = *(const u32x4 *)(stage + br * EPI_Z_STRIDE + hpiece * 16);
                    *(u32x4 *)(a.aux2 + (row0 + wq + i * 32 + br) * a.ldaux2 + ch) = v;
                }
                wave_lds_sync();
            }
        }
        };
        blocks(IC<epi_scaled_act(EPI) ? 1 : 0>{});
    }
}

} // namespace xma_rocm
