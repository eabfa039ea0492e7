// gemm_group.h -- many GEMM problems in one launch: grouped and served
// requests, rank-k updates, the tile runtime's rounds.  Instantiated per
// element type (gemm_group_{s,d,z}.hip).
//
// A block finds its problem by its tile number and runs one block tile of it
// (gemm_tile.h).  k_group holds the 64x64 and 32x32 tiles, both ways of
// moving operands and every transpose: 32 KB of LDS and at most 168 registers,
// three blocks on a CU.  k_group_big holds the 128x64 and (real types) 128x128
// tiles of 16-byte aligned operands, for launches that fill the GPU many times over
// (FP64, one 8192^3 product: 76 TFLOP/s on either, 70 on 64x64).
#pragma once
#include "gemm_tile.h"

namespace {

// The problem of tile t: the last whose tile_start is <= t.  64 lanes probe 64
// problems at a time, so that the chain of dependent loads before a block's
// first operand load is one or two long.
__device__ __forceinline__ int find_problem(const bxh_problem_t *__restrict__ probs, int nprob, int t)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = nprob; // the answer is in [lo, hi)
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) / 64, i = lo + lane * step;
        const bool le = i < hi && probs[i].tile_start <= t;
        const int c = __builtin_popcountll(__ballot(le)); // >= 1: probs[lo] is
        lo += (c - 1) * step;
        hi = min(hi, lo + step);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

template <typename E, int WTM, int WTN, int NS, bool DMA, int G>
__device__ __forceinline__ void group_tile(const bxh_problem_t &P, const bxh_seg_t *segs, int local,
                                           char *smem)
{
    typedef Shape<E, WTM, WTN, NS> H;
    int tm, tn;
    if constexpr (Shape<E, WTM, WTN, NS>::BM == 128)
        tile_coords_striped<G>(local, P.tiles_m, P.tiles_n, tm, tn);
    else
        tile_coords<G>(local, P.tiles_m, P.tiles_n, tm, tn);
    if (P.tri) {
        // a tile of a rank-k diagonal block wholly off the stored triangle
        const int r0 = tm * H::BM + P.tri_off, c0 = tn * H::BN;
        if ((P.tri & BX_TRI_LOWER) && r0 + H::BM - 1 < c0) return;
        if ((P.tri & BX_TRI_UPPER) && r0 > c0 + H::BN - 1) return;
    }
    const bxh_seg_t unused = {nullptr, nullptr, 0, 0, 0};
#define BX_TILE(MA_, MB_, CA_, CB_)                                                                \
    tile_block<E, MA_, MB_, CA_, CB_, WTM, WTN, NS, DMA>(P, segs, unused, unused, tm, tn, smem);   \
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

// counts != NULL: graph replay, the problem count and the tile total are
// read from device memory (counts[0], counts[1]) and the grid is fixed
template <typename E>
__global__ __launch_bounds__(NT, 3) void k_group(const bxh_problem_t *__restrict__ probs, int nprob,
                                                 const bxh_seg_t *__restrict__ segs, int total,
                                                 const int *__restrict__ counts)
{
    __shared__ __attribute__((aligned(16))) char smem[Shape<E, 32, 32, 2>::SMEM];
    static_assert(Shape<E, 16, 16, 4>::SMEM == Shape<E, 32, 32, 2>::SMEM, "one LDS size");
    if (counts) {
        nprob = counts[0];
        total = counts[1];
    }
    for (int t = blockIdx.x; t < total; t += gridDim.x) {
        const bxh_problem_t P = probs[find_problem(probs, nprob, t)];
        const bxh_seg_t *ps = segs + P.seg_off;
        const int local = t - P.tile_start;
        if (P.shape == BXH_SHAPE_32x32) {
            if (P.form == BXH_FORM_DMA) group_tile<E, 16, 16, 4, true, 8>(P, ps, local, smem);
            else group_tile<E, 16, 16, 2, false, 8>(P, ps, local, smem);
        } else {
            if (P.form == BXH_FORM_DMA) group_tile<E, 32, 32, 2, true, 8>(P, ps, local, smem);
            else group_tile<E, 32, 32, 2, false, 8>(P, ps, local, smem);
        }
        __syncthreads(); // the next tile reuses the stages
    }
}

template <typename E>
__global__ __launch_bounds__(NT, 2) void k_group_big(const bxh_problem_t *__restrict__ probs,
                                                     int nprob, const bxh_seg_t *__restrict__ segs)
{
    __shared__ __attribute__((aligned(16))) char smem[Shape<E, 64, 64, 2>::SMEM];
    const int t = blockIdx.x;
    const bxh_problem_t P = probs[find_problem(probs, nprob, t)];
    const bxh_seg_t *ps = segs + P.seg_off;
    if constexpr (sizeof(E) != 16)
        if (P.shape == BXH_SHAPE_128x128) {
            group_tile<E, 64, 64, 2, true, 4>(P, ps, t - P.tile_start, smem);
            return;
        }
    group_tile<E, 64, 32, 2, true, 4>(P, ps, t - P.tile_start, smem);
}

template <typename E>
int launch_group(const bxh_problem_t *probs, int nprob, const bxh_seg_t *segs, int total, int grid,
                 const int *counts, hipStream_t st)
{
    if (grid == BXH_GROUP_BIG) {
        hipLaunchKernelGGL(k_group_big<E>, dim3(total), dim3(NT), 0, st, probs, nprob, segs);
    } else {
        if (grid <= 0 || (!counts && grid > total)) grid = total;
        // a grid's threads fit 32 bits: beyond, blocks take several tiles
        if (grid >= (1 << 24)) grid = (1 << 24) - 1;
        hipLaunchKernelGGL(k_group<E>, dim3(grid), dim3(NT), 0, st, probs, nprob, segs, total, counts);
    }
    return bx_launch_status("grouped gemm launch");
}

} // namespace
