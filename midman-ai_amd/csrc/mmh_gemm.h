// Shared by the GEMM kernels: the launch parameters and the few device helpers
// that both the small-tile kernels (gemm.hip) and the large-tile kernels
// (gemm_split.hip) use.
#pragma once

#include "mmh_internal.h"

namespace mmh {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// Raw buffer descriptor: byte range (interior tiles stay below 2^31 bytes from
// their base, checked on the host) and the gfx9-family dword-3 flags.
constexpr int kBufferRange = 0x7fffffff;
constexpr int kBufferFlags = 0x00020000;

// The loss partials come one per 128 columns; K advances 16 at a time in the
// large-tile kernels.
constexpr int BM = 128, BN = 128, BK = 16;

struct KParams {
    const float *a;
    const float *b;
    float *c;
    float *partial;
    int64_t m, n, k;
    int64_t lda, ldb, ldc;
    int64_t stride_a, stride_b, stride_c;
    int64_t k_per_split;
    int64_t swiglu_ff;
    const float *resid;
    float *aux;
    int64_t ldaux;
    int tiles_m, tiles_n;
    int splits;
    int vec_a, vec_b, vec_c;
    // small kernel only: A-row RMSNorm in the loads, RoPE in the epilogue
    const float *norm_w;
    float norm_eps;
    const float *rope_cos, *rope_sin;
    int rope_seq, rope_hd, rope_cols;
    // EPI_CE (large tiles): targets in, (max, sum) pairs per 128 columns and target logits out
    const int32_t *ce_targets;
    float *ce_part, *ce_zt;
    int ce_tiles;  // 128-column units of a row
    // Large tiles, the exponentials of EPI_SWIGLU and EPI_CE: libm's (and the IEEE
    // division) where the grid has less than a 128x128 tile per CU, as the small
    // kernels have it. The hardware's exp2 of a rounded product, which fuller
    // grids take, is off by |x| 2^-24 of itself: gates of -60 to -40 give h off by
    // 3.3e-6, 3.0e-7 by libm's. libm's costs 1-3% of a model's loss there (8 layers
    // of 768, 512 tokens: 1079 -> 1093 us).
    int libm_exp;
    // Split K on the 64x64 and 32x32 tiles (tickets set): every split stores
    // its partial tile through to memory and counts itself in tickets[tile];
    // the last split of a tile sums the tile's partials in split order and
    // applies the epilogue (split_accum: C = resid (or C) + sum, else C = sum).
    int32_t *tickets;
    int split_accum;
    // The value the sums of products start from: +0 (a product, as the
    // reference's fresh zeroed C), or -0 when the sum is added into C (the
    // seam's accumulate: C's own value starts the reference's sum, so a -0 in
    // C with all products -0 must stay -0; -0 is the identity of IEEE addition)
    float acc_init;
};


// ---- gemm_split.hip ---------------------------------------------------------

// Tile shapes of the large-tile kernels: rows x columns, and the groups of
// waves that share a tile's K.
enum GemmTile : int { TILE_256, TILE_256x128, TILE_128, TILE_128x64, TILE_64, TILE_COUNT };
struct GemmTileInfo {
    int rows, cols;
    // us per 16 of K on an MI355X: a workgroup that has its CU to itself, and
    // the share of a chip with one on every CU, where its power sets the rate;
    // and the first loads and the epilogue of a tile in such steps (choose_tile)
    float alone, full, setup;
};
constexpr GemmTileInfo kGemmTiles[TILE_COUNT] = {
    {256, 256, 1.75f, 2.35f, 7.5f}, {256, 128, 1.0f, 1.29f, 6.0f}, {128, 128, 0.55f, 0.72f, 10.0f},
    {128, 64, 0.42f, 0.43f, 8.0f},  {64, 64, 0.25f, 0.26f, 14.0f},
};
// The tile kernel for p's product in the given form and epilogue; p.tiles_m and
// p.tiles_n count tiles of the given shape. Splits (grid z) write their sums
// to p.partial; launch_splitk_reduce adds them in split order.
bool gemm_tile_takes(const KParams &p, int epi, int tile);
void launch_gemm_tiles(Context &ctx, const KParams &p, dim3 grid, bool ta, bool tb, int epi,
                       int tile);
void launch_splitk_reduce(Context &ctx, const KParams &p, int epi);

}  // namespace mmh
