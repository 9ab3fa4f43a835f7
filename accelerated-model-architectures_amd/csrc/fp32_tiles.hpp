// Which tile an fp32 GEMM takes, of 64 x 64 or 128 x 128 outputs (fp32.hip); plain C++, so that a test can ask on the host.  The small one
// pays where the large ones leave compute units idle, below two per unit, and where they are padding by more than the small one's extra traffic
// through LDS is worth.  Results are bit-identical.
#pragma once

#include <math.h>
#include <stdint.h>

constexpr int f32_tile_step(int dim) { return dim == 64 ? 32 : 16; } // of K: the tile's two operands take 16 KB
inline int64_t f32_tiles(int64_t m, int64_t n, int dim) { return ((m + dim - 1) / dim) * ((n + dim - 1) / dim); }
inline double f32_padded(int64_t n, int dim) { return (double)((n + dim - 1) / dim * dim); }
// rows that tiles of `dim` multiply for an expert of about `rows` (within two standard deviations of a random load): an expert ends in half a
// tile on average
inline double f32_padded_load(double rows, int dim) {
    const double lo = ceil((rows - 2 * sqrt(rows)) / dim), hi = ceil((rows + 2 * sqrt(rows)) / dim);
    return dim * (lo == hi ? hi : rows / dim + 0.5);
}

// Forward / dX.  Large / small tile in us (x @ W^T; dy @ W).  Rows: 64 experts of K = 1024, N = 2048, 30 rows each 287 / 162;
// 286 / 166, 90 rows (one large tile or two) 303 / 325; 296 / 339; 128 of K = 576, N = 512, 125 rows 128 / 114; 127 / 116, 250 rows 212 /
// 199; 207 / 202, 500 rows 379 / 378; 367 / 372, 1000 rows 689 / 706; 677 / 710; 30 of K = 400, N = 1200, 300 rows 122 / 99; 121 / 102; 16 of
// K = 1024, N = 4096, 250 rows 352 / 326; 350 / 340.  Tiles: 8 experts of K = 2048, N = 512, 256 tiles 168 / 150; 174 / 155, 512 of them 293 /
// 295; 284 / 299, of K = 512, N = 2048, 4096 tiles 563 / 602; 558 / 622.  A short K is padded as well: 64 experts of 115 rows, K = 72 (80 / 96), N =
// 1376 37 / 44; of 45, 346 rows, K = 112, N = 1456 91 / 99.
inline bool f32_small_tile(int64_t M, int64_t N, int64_t K, int64_t E) {
    auto work = [&](int dim) { return f32_padded_load((double)M / E, dim) * f32_padded(N, dim) * f32_padded(K, f32_tile_step(dim)); };
    return E * f32_tiles((M + E - 1) / E, N, 128) < 512 || 1.04 * work(64) < work(128);
}

// dW, whose reduction is the expert's rows: M of them in all, 0 where nobody knows.  8 experts of 500 rows, 256 tiles 62 / 52, 512 tiles
// 96 / 109; 1000 x 2048 x 2048 4 experts 309 / 343; 128 of 576 x 512, 500 rows 413 / 427; padded by a fifth, 30 of 1200 x 400, 300 rows 141 /
// 116, 700 rows 285 / 251.  With few rows a launch is its stores, and those of a large tile are whole lines: 45 experts of 3568 x 424 (0.88 of
// the large tiles' padding), 10 rows 66 / 91; 128 of 448 x 1080 (0.83), 2 rows 51 / 68; from 32 rows on 0.5 - 0.95 of the time.
inline bool f32_small_tile_dw(int64_t M, int64_t N_out, int64_t K_in, int64_t E) {
    const double worse = M > 0 ? 1.12 + 2. * E / M : 1.43; // 0.7 of the padding is less than the large tiles' at any number of rows
    return E * f32_tiles(N_out, K_in, 128) < 512 ||
           worse * f32_padded(N_out, 64) * f32_padded(K_in, 64) < f32_padded(N_out, 128) * f32_padded(K_in, 128);
}
