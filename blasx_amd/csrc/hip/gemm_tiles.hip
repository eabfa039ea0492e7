// gemm_tiles.hip -- one product per launch on the block tile shape that runs
// it fastest (gemm_tile.h).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../tilecost.h"
#include "gemm_tile.h"

namespace {

// Tile rows walked together.  An XCD's blocks start in step but drift apart in
// K, so that long products lose the panel sharing in its L2; what the walk
// keeps is what the Infinity Cache serves.  32768^3, FP64, 128x128 tiles: each
// XCD on a contiguous range of groups of 4 rows 75.8 TFLOP/s, all XCDs striped
// over one group 76.1; rank-k updates (N = K = 32768): ranges 69.2, striped
// groups of 8, 4 and 2 rows 69.8, 71.1 and 71.7 (complex, 128x64 tiles: 2 rows
// 75.3, ranges 73.9).  Shorter products keep ranges: 8192^3 on 128x64 tiles
// reaches 76.1 with groups of 4 rows, 73.4 with 8.
constexpr int G_SMALL = 8, G_BIG = 4, G_TRI = 2;

// S1: the second K segment of a rank-2k update
template <typename E, int MAJA, int MAJB, bool CJA, bool CJB, int WTM, int WTN, int NS, bool DMA, int OCC>
__global__ __launch_bounds__(NT, OCC) void k_tile(bxh_problem_t P, bxh_seg_t S, bxh_seg_t S1)
{
    typedef Shape<E, WTM, WTN, NS> H;
    __shared__ __attribute__((aligned(16))) char smem[H::SMEM];
    int tm, tn;
    if (P.tri) {
        tri_coords<G_TRI, H::BM, H::BN>(blockIdx.x, P.tri & BX_TRI_UPPER, P.tiles_m, P.tiles_n, tm, tn);
        // a tile wholly off the stored triangle
        const int r0 = tm * H::BM, c0 = tn * H::BN;
        if ((P.tri & BX_TRI_LOWER) && r0 + H::BM - 1 < c0) return;
        if ((P.tri & BX_TRI_UPPER) && r0 > c0 + H::BN - 1) return;
    } else if constexpr (H::BM * H::BN == 128 * 128) {
        tile_coords_striped<G_BIG>(blockIdx.x, P.tiles_m, P.tiles_n, tm, tn);
    } else {
        tile_coords<H::BM == 128 ? G_BIG : G_SMALL>(xcd_tile(), P.tiles_m, P.tiles_n, tm, tn);
    }
    tile_block<E, MAJA, MAJB, CJA, CJB, WTM, WTN, NS, DMA>(P, nullptr, S, S1, tm, tn, smem);
}

// A launch's threads fit 32 bits along a dimension, and a tile's rows an int.
// Skinny products of hundreds of millions of columns would have more tiles
// of 32x32 (or 64 rows) than that.
constexpr int64_t MOST_TILES = ((int64_t)1 << 32) / NT - 1;
constexpr int MOST_ROWS = INT32_MAX - 127;

template <int BM, int BN> int64_t grid_tiles(int tri, int m, int n)
{
    const int tm = (m + BM - 1) / BM, tn = (n + BN - 1) / BN;
    return tri ? tri_tiles<G_TRI, BM, BN>(tm, tn) : (int64_t)tm * tn;
}
int64_t shape_tiles(int s, int tri, int m, int n)
{
    switch (s) {
    case BXC_32x32: return grid_tiles<32, 32>(tri, m, n);
    case BXC_64x32: return grid_tiles<64, 32>(tri, m, n);
    case BXC_64x64: return grid_tiles<64, 64>(tri, m, n);
    case BXC_128x64: return grid_tiles<128, 64>(tri, m, n);
    default: return grid_tiles<128, 128>(tri, m, n);
    }
}

template <typename E, int WTM, int WTN, int NS, bool DMA, int OCC>
void launch_shape(bxh_problem_t P, const bxh_seg_t *S, hipStream_t st)
{
    typedef Shape<E, WTM, WTN, NS> H;
    P.tiles_m = (P.m + H::BM - 1) / H::BM;
    P.tiles_n = (P.n + H::BN - 1) / H::BN;
    const dim3 grid((unsigned)grid_tiles<H::BM, H::BN>(P.tri, P.m, P.n));
    const bxh_seg_t S0 = S[0], S1 = S[P.nseg > 1];
#define BX_TILE(MA_, MB_, CA_, CB_)                                                              \
    hipLaunchKernelGGL((k_tile<E, MA_, MB_, CA_, CB_, WTM, WTN, NS, DMA, OCC>), grid, dim3(NT), 0, st, \
                       P, S0, S1);                                                                    \
    break
    if constexpr (sizeof(E) == 16) {
        switch (P.opa * 3 + P.opb) {
        case 0: BX_TILE(MAJ_MN, MAJ_K, false, false);
        case 1: BX_TILE(MAJ_MN, MAJ_MN, false, false);
        case 2: BX_TILE(MAJ_MN, MAJ_MN, false, true);
        case 3: BX_TILE(MAJ_K, MAJ_K, false, false);
        case 4: BX_TILE(MAJ_K, MAJ_MN, false, false);
        case 5: BX_TILE(MAJ_K, MAJ_MN, false, true);
        case 6: BX_TILE(MAJ_K, MAJ_K, true, false);
        case 7: BX_TILE(MAJ_K, MAJ_MN, true, false);
        default: BX_TILE(MAJ_K, MAJ_MN, true, true);
        }
    } else {
        switch ((P.opa != 0) * 2 + (P.opb != 0)) {
        case 0: BX_TILE(MAJ_MN, MAJ_K, false, false);
        case 1: BX_TILE(MAJ_MN, MAJ_MN, false, false);
        case 2: BX_TILE(MAJ_K, MAJ_K, false, false);
        default: BX_TILE(MAJ_K, MAJ_MN, false, false);
        }
    }
#undef BX_TILE
}

} // namespace

namespace {

// the shape that runs one product fastest (tilecost.h; all tiles alike, so
// the busiest CU has the rounded-up share) in at most `most` tiles; the
// largest tile where none does
int best_shape(int dtype, bool dma, int tri, int m, int n, int64_t k, int64_t most)
{
    int best = BXC_32x32;
    double bt = 1e300;
    for (int s = BXC_32x32; s < BXC_SHAPES; ++s) {
        const bx_cost_t &c = dma ? BX_COST_DMA[dtype][s] : BX_COST_REG[dtype][s];
        if (c.a <= 0) continue;
        const int64_t tiles = shape_tiles(s, tri, m, n);
        if (bt == 1e300) best = s;
        if (tiles > most) continue;
        const double t = c.l + (double)((tiles + 255) / 256) * bx_cost_tile(&c, k);
        if (t < bt) {
            bt = t;
            best = s;
        }
    }
    return best;
}

// false: no such tile for this type and form
template <typename E>
bool launch_tile(int s, const bxh_problem_t &P, const bxh_seg_t *S, hipStream_t st)
{
    if (P.form != BXH_FORM_DMA) {
        switch (s) {
        case BXC_32x32: launch_shape<E, 16, 16, 2, false, 4>(P, S, st); return true;
        case BXC_64x32: launch_shape<E, 32, 16, 2, false, 4>(P, S, st); return true;
        case BXC_64x64: launch_shape<E, 32, 32, 2, false, 3>(P, S, st); return true;
        }
        return false;
    }
    switch (s) {
    case BXC_32x32: launch_shape<E, 16, 16, 4, true, 4>(P, S, st); return true;
    case BXC_64x32: launch_shape<E, 32, 16, 4, true, 3>(P, S, st); return true;
    case BXC_64x64: launch_shape<E, 32, 32, 4, true, 2>(P, S, st); return true;
    case BXC_128x64:
        launch_shape<E, 64, 32, sizeof(E) == 16 ? 2 : 3, true, 2>(P, S, st);
        return true;
    }
    if constexpr (sizeof(E) == 8)
        if (s == BXC_128x128) {
            launch_shape<E, 64, 64, 2, true, 2>(P, S, st);
            return true;
        }
    return false;
}

} // namespace

extern "C" {

int bxh_gemm_tile_most(int dtype, int shape, const bxh_problem_t *P, const bxh_seg_t *S, void *stream,
                       int64_t most)
{
    if (dtype < 0 || dtype > 2 || P->nseg < 1 || P->nseg > 2 || (P->tri && P->m != P->n))
        return BLASX_EINVAL;
    const int big = P->m > P->n ? P->m : P->n;
    bxh_problem_t Q = *P;
    Q.form = BXH_FORM_DMA;
    int64_t k = 0;
    for (int i = 0; i < P->nseg; ++i) {
        const int f = bxh_tile_form(dtype, P->opa, P->opb, P->m, P->n, &S[i]);
        Q.form = f > Q.form ? f : Q.form;
        k += S[i].k;
    }
    int s = shape;
    if (big <= MOST_ROWS) {
        if (s < 0) s = best_shape(dtype, Q.form == BXH_FORM_DMA, P->tri, P->m, P->n, k, most);
        if (s >= BXC_SHAPES) return BLASX_EINVAL;
    }
    if (!P->tri && big > 128 && (big > MOST_ROWS || shape_tiles(s, 0, P->m, P->n) > most)) {
        // too many tiles for one launch: the longer side in halves
        const int es = dtype == BLASX_S ? 4 : dtype == BLASX_D ? 8 : 16;
        const bool rows = P->m == big;
        const int64_t h = ((int64_t)big / 2 + 127) / 128 * 128;
        bxh_seg_t S2[2];
        for (int i = 0; i < P->nseg; ++i) {
            S2[i] = S[i];
            if (rows)
                S2[i].A = (const char *)S[i].A + (P->opa == 0 ? h : h * S[i].lda) * es;
            else
                S2[i].B = (const char *)S[i].B + (P->opb == 0 ? h * S[i].ldb : h) * es;
        }
        (rows ? Q.m : Q.n) = (int)h;
        const int rc = bxh_gemm_tile_most(dtype, shape, &Q, S, stream, most);
        if (rc) return rc;
        (rows ? Q.m : Q.n) = big - (int)h;
        Q.C = (char *)P->C + (rows ? h : h * P->ldc) * es;
        return bxh_gemm_tile_most(dtype, shape, &Q, S2, stream, most);
    }
    hipStream_t st = (hipStream_t)stream;
    const bool ran = dtype == BLASX_S   ? launch_tile<float>(s, Q, S, st)
                     : dtype == BLASX_D ? launch_tile<double>(s, Q, S, st)
                                        : launch_tile<cplx>(s, Q, S, st);
    if (!ran) return BLASX_EINVAL;
    return bx_launch_status(P->tri ? "rank-k launch" : "gemm launch");
}

int bxh_gemm_tile_as(int dtype, int shape, const bxh_problem_t *P, const bxh_seg_t *S, void *stream)
{
    return bxh_gemm_tile_most(dtype, shape, P, S, stream, MOST_TILES);
}

int bxh_gemm_tile(int dtype, const bxh_problem_t *P, const bxh_seg_t *S, void *stream)
{
    return bxh_gemm_tile_as(dtype, -1, P, S, stream);
}

// for the test-suite: the tile of block t of a launch of a shape's tiles (tri:
// BX_TRI_* bits, the triangular walk; else the striped one), false past the
// grid; and the shape (BXC_*) that bxh_gemm_tile takes
int bxh_tile_at_host(int shape, int tri, int m, int n, int64_t t, int *tm, int *tn)
{
    const int tiles_m = (m + BX_COST_BM[shape] - 1) / BX_COST_BM[shape];
    const int tiles_n = (n + BX_COST_BN[shape] - 1) / BX_COST_BN[shape];
    if (t >= shape_tiles(shape, tri, m, n)) return 0;
    if (!tri) {
        tile_coords_striped<G_BIG>((int)t, tiles_m, tiles_n, *tm, *tn);
        return 1;
    }
    const int up = tri & BX_TRI_UPPER;
    switch (shape) {
    case BXC_32x32: tri_coords<G_TRI, 32, 32>(t, up, tiles_m, tiles_n, *tm, *tn); break;
    case BXC_64x32: tri_coords<G_TRI, 64, 32>(t, up, tiles_m, tiles_n, *tm, *tn); break;
    case BXC_64x64: tri_coords<G_TRI, 64, 64>(t, up, tiles_m, tiles_n, *tm, *tn); break;
    case BXC_128x64: tri_coords<G_TRI, 128, 64>(t, up, tiles_m, tiles_n, *tm, *tn); break;
    default: tri_coords<G_TRI, 128, 128>(t, up, tiles_m, tiles_n, *tm, *tn);
    }
    return 1;
}
int bxh_tile_shape_host(int dtype, int dma, int tri, int m, int n, int64_t k)
{
    return best_shape(dtype, dma != 0, tri, m, n, k, MOST_TILES);
}

} // extern "C"
