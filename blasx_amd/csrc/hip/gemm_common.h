// gemm_common.h -- element types, MFMA forms, epilogue arithmetic and tile
// walk shared by the GEMM kernels (gemm_kernels.hip, gemm_tiles.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../hiplayer.h"
#include "blasx_ext.h"
#include "gmem.h"

// 0, or BLASX_EHIP with the launch's own error kept for bxh_last_error
// (gemm_kernels.hip)
extern "C" int bx_launch_status(const char *what);

namespace {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

struct cplx {
    double re, im;
};

template <typename E> struct Cfg;
// OUT_ROW(lg, v): the 16x16 MFMA output row held by accumulator element v
// of a lane in lane-group lg = lane / 16 (column = lane % 16).  Measured on
// gfx950: the FP32 16x16x4 MFMA returns rows 4*lg + v, the FP64 16x16x4
// MFMA returns rows lg + 4*v.
template <> struct Cfg<double> {
    static constexpr int BM = 128, BN = 128;
    typedef d4_t acc_t;
    static __device__ __forceinline__ int out_row(int lg, int v) { return lg + 4 * v; }
};
template <> struct Cfg<float> {
    static constexpr int BM = 128, BN = 128;
    typedef f4_t acc_t;
    static __device__ __forceinline__ int out_row(int lg, int v) { return 4 * lg + v; }
};
template <> struct Cfg<cplx> {
    static constexpr int BM = 128, BN = 64;
    typedef d4_t acc_t;
    static __device__ __forceinline__ int out_row(int lg, int v) { return lg + 4 * v; }
};

constexpr int NT = 256;
enum { MAJ_MN = 0, MAJ_K = 1 };

template <typename E> __device__ __forceinline__ E zero_of() { return E(0); }
template <> __device__ __forceinline__ cplx zero_of<cplx>() { return cplx{0.0, 0.0}; }

// The epilogue's arithmetic, one rounding sequence for every kernel (explicit
// FMAs: no result depends on how the compiler contracts a kernel's code).
// alpha * s, then + beta * c in one FMA; c is not used when beta_zero.
template <typename E>
__device__ __forceinline__ E out_real(E alpha, E s, E beta, E c, bool beta_zero)
{
    const E x = alpha * s;
    return beta_zero ? x : fma(beta, c, x);
}
// complex: alpha (sr + i sim), then + beta c
__device__ __forceinline__ cplx out_cplx(double ar, double ai, double sr, double sim, double br,
                                         double bi, cplx c, bool beta_zero)
{
    double orr = fma(ar, sr, -(ai * sim)), oi = fma(ar, sim, ai * sr);
    if (!beta_zero) {
        orr = fma(br, c.re, fma(-bi, c.im, orr));
        oi = fma(br, c.im, fma(bi, c.re, oi));
    }
    return cplx{orr, oi};
}

__device__ __forceinline__ d4_t mfma(double a, double b, d4_t c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma(float a, float b, f4_t c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__host__ __device__ __forceinline__ bool aligned16(const void *p, int64_t ld, int esize)
{
    return ((reinterpret_cast<uintptr_t>(p) & 15) == 0) && (((ld * esize) & 15) == 0);
}

// Tile loc of a group of `rows` tile rows and `cols` tile columns, walked so
// that all XCDs (block b runs on XCD b % 8) are on the same rows, each on
// columns of its own: the rows' operand panels come from the Infinity Cache
// whatever K each block has reached, and a column's panel is read by the
// `rows` blocks that one XCD runs one after the other.
__host__ __device__ __forceinline__ void striped(int64_t loc, int rows, int cols, int &r, int &c)
{
    const int full = cols & ~7;
    const int64_t nf = (int64_t)rows * full;
    if (loc < nf) {
        const int64_t q = loc >> 3;
        r = (int)(q % rows);
        c = (int)(q / rows) * 8 + (int)(loc & 7);
    } else {
        const int w = cols - full;
        r = (int)((loc - nf) / w);
        c = full + (int)((loc - nf) % w);
    }
}
template <int G>
__host__ __device__ __forceinline__ void tile_coords_striped(int t, int tiles_m, int tiles_n, int &tm,
                                                             int &tn)
{
    const int64_t per = (int64_t)G * tiles_n;
    const int g = (int)(t / per), rows = tiles_m - g * G < G ? tiles_m - g * G : G;
    int r;
    striped(t - g * per, rows, tiles_n, r, tn);
    tm = g * G + r;
}

// The tiles of a rank-k update's stored triangle, G tile rows at a time, each
// group striped over the XCDs: group g has its first tri_cols(g) tile columns
// (for an upper triangle, both counted from the last).  The few tiles of a
// group beyond the diagonal are skipped by the kernel.
template <int G, int BM, int BN> __host__ __device__ __forceinline__ int64_t tri_cols(int64_t g, int tiles_n)
{
    static_assert(BM % BN == 0, "whole columns per row");
    const int64_t c = (BM / BN) * G * (g + 1) + 1;
    return c < tiles_n ? c : tiles_n;
}
// tiles before group g (only the last group's columns can be clipped: a group
// before it ends at least one column short of the last)
template <int G, int BM, int BN> __host__ __device__ __forceinline__ int64_t tri_before(int64_t g)
{
    return G * ((BM / BN) * G * (g * (g + 1) / 2) + g);
}
template <int G, int BM, int BN>
__host__ __device__ __forceinline__ int64_t tri_tiles(int tiles_m, int tiles_n)
{
    const int64_t last = (tiles_m - 1) / G;
    return tri_before<G, BM, BN>(last) + (tiles_m - last * G) * tri_cols<G, BM, BN>(last, tiles_n);
}
template <int G, int BM, int BN>
__host__ __device__ __forceinline__ void tri_coords(int64_t t, int upper, int tiles_m, int tiles_n,
                                                    int &tm, int &tn)
{
    // g: the last group that starts at or before t
    const double r = (BM / BN) * (double)G * G, h = r / 2 + G;
    int64_t g = (int64_t)((sqrt(h * h + 2 * r * (double)t) - h) / r);
    while (g > 0 && tri_before<G, BM, BN>(g) > t) --g;
    while (tri_before<G, BM, BN>(g + 1) <= t) ++g;
    const int64_t last = (tiles_m - 1) / G;
    if (g > last) g = last;
    const int rows = (int)(tiles_m - g * G < G ? tiles_m - g * G : G);
    int row;
    striped(t - tri_before<G, BM, BN>(g), rows, (int)tri_cols<G, BM, BN>(g, tiles_n), row, tn);
    tm = (int)g * G + row;
    if (upper) {
        tm = tiles_m - 1 - tm;
        tn = tiles_n - 1 - tn;
    }
}

// block tile index -> (tm, tn), walking groups of 8 tile rows so that the
// blocks resident at one time share A row panels and B column panels
template <int G = 8>
__device__ __forceinline__ void tile_coords(int t, int tiles_m, int tiles_n, int &tm, int &tn)
{
    const int per_group = G * tiles_n;
    const int g = t / per_group;
    const int first = g * G;
    const int gsz = min(tiles_m - first, G);
    const int r = t - g * per_group;
    tm = first + r % gsz;
    tn = r / gsz;
}

// segment i of the table, or of the by-value pair when there is no table;
// fields are read through the global address space one by one (selecting
// between a table pointer and a local would make every access FLAT)
__device__ __forceinline__ bxh_seg_t seg_at(const bxh_seg_t *segs, const bxh_seg_t &seg0,
                                            const bxh_seg_t &seg1, int i)
{
    bxh_seg_t s;
    if (!segs) {
        s.A = i ? seg1.A : seg0.A;
        s.B = i ? seg1.B : seg0.B;
        s.lda = i ? seg1.lda : seg0.lda;
        s.ldb = i ? seg1.ldb : seg0.ldb;
        s.k = i ? seg1.k : seg0.k;
        return s;
    }
    const __attribute__((address_space(1))) bxh_seg_t *g =
        (const __attribute__((address_space(1))) bxh_seg_t *)(segs + i);
    s.A = g->A;
    s.B = g->B;
    s.lda = g->lda;
    s.ldb = g->ldb;
    s.k = g->k;
    return s;
}

// whether a rank-k update writes element (row, col) of its diagonal block
__device__ __forceinline__ bool tri_keep(int tri, int row, int col)
{
    return (!(tri & BX_TRI_LOWER) || row >= col) && (!(tri & BX_TRI_UPPER) || row <= col);
}


} // namespace
