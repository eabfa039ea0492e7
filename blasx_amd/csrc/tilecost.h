/*
 * tilecost.h -- estimated launch times of the GEMM block tile shapes, for
 * picking one (hip/gemm_tiles.hip, grouped.c, syrk.c, tile_rt.c).
 *
 * A launch of `tiles` equal tiles of a shape over K takes about l + n (c +
 * a K / 1000) microseconds, n = tiles of the busiest of the 256 CUs: a = one
 * tile's time per 1000 of K (the matrix core's rate, and at the small shapes
 * what LDS and L2 leave of it), c = its start and its writes of C.  Fitted to
 * launch times of random products (M, N, K log-uniform in 64..8192; 80 to 110
 * per row; the choice was 1-2% slower than the best shape on average), the
 * rows of the 64x64 and larger tiles then moved by up to 2% so that products
 * above 4096^3, few in the fit, go to the 128-row tiles that run them faster.
 * The complex rows: 640 products and triangles up to 32768, the coefficients
 * then searched for the least loss of the choice against each product's fastest
 * shape (on average 0.5% on large and mid-sized products, 0.2% on small ones, 0.5
 * to 1% on triangles).  What 64x32 tiles lose beyond K = 2048 and 64x64 ones in
 * wide triangles is L2 misses (8192^3: 32x32 62, 64x32 70, 64x64 76.4, 128x64
 * 76.9 TFLOP/s; a triangle of 16384, K = 8192: 59, 70, 69.5 and 74.8), so l of
 * 128x64 is what keeps products too short for that on finer tiles, not a time.
 * Measured rates at 4096^3, FP64: 32x32 57, 64x32 69, 64x64 74.5, 128x64 75
 * TFLOP/s; at 8192^3, where L2 misses count, 64x64 70, 128x64 and 128x128 76;
 * but 1024^3 takes 35, 34, 34 and 66 us on the first four, 256^3 5, 7, 11, 19.
 */
#ifndef BLASX_TILECOST_H
#define BLASX_TILECOST_H

#include <stdint.h>

enum { BXC_32x32, BXC_64x32, BXC_64x64, BXC_128x64, BXC_128x128, BXC_SHAPES };

typedef struct {
    float l, c, a; /* a <= 0: no such tile, or (FP32 128x128) never a better one */
} bx_cost_t;

static const int BX_COST_BM[BXC_SHAPES] = {32, 64, 64, 128, 128};
static const int BX_COST_BN[BXC_SHAPES] = {32, 32, 64, 64, 128};
/* by element type (S, D, Z): operands by DMA, and through registers */
static const bx_cost_t BX_COST_DMA[3][BXC_SHAPES] = {
    {{3.0f, 0.53f, 3.99f}, {3.4f, 0.88f, 7.39f}, {3.8f, 1.71f, 14.9f}, {5.7f, 4.5f, 29.3f}, {0, 0, 0}},
    {{2.5f, 0.56f, 7.75f}, {3.0f, 0.87f, 14.39f}, {3.7f, 1.69f, 28.4f}, {5.6f, 2.19f, 56.6f}, {5.6f, 9.0f, 112.6f}},
    {{0.5f, 0.75f, 30.2f}, {8.2f, 0.80f, 56.8f}, {10.5f, 2.45f, 111.1f}, {130.0f, 2.2f, 214.0f}, {0, 0, 0}},
};
static const bx_cost_t BX_COST_REG[3][BXC_SHAPES] = {
    {{3.5f, 0.39f, 5.04f}, {3.7f, 0.72f, 9.05f}, {4.3f, 1.21f, 17.4f}, {0, 0, 0}, {0, 0, 0}},
    {{3.1f, 0.30f, 10.04f}, {3.7f, 0.47f, 17.8f}, {4.2f, 1.18f, 33.4f}, {0, 0, 0}, {0, 0, 0}},
    {{2.4f, 0.50f, 32.5f}, {6.9f, 1.01f, 61.8f}, {14.4f, 0.05f, 123.0f}, {0, 0, 0}, {0, 0, 0}},
};

static inline int64_t bx_cost_tiles(int s, int m, int n)
{
    return (int64_t)((m + BX_COST_BM[s] - 1) / BX_COST_BM[s]) * ((n + BX_COST_BN[s] - 1) / BX_COST_BN[s]);
}

/* Tiles of the busiest CU in a grouped launch of tiles up to 64x64, three of which
 * share a CU: just beyond 768 the second round falls on whichever CUs finish
 * first (1024 tiles, K = 2048: FP64 316 us and complex 1134, as long as five a
 * CU); later rounds even out (4096 tiles: 15.7 a CU). */
static inline int64_t bx_cost_group_busiest(int64_t tiles)
{
    return (tiles + 255) / 256 + (tiles > 768 && tiles <= 1280);
}

/* one tile's time */
static inline double bx_cost_tile(const bx_cost_t *c, int64_t k) { return c->c + c->a * 1e-3 * (double)k; }

#endif
