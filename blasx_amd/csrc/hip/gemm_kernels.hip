// gemm_kernels.hip -- entry points of the GEMM launches (one problem:
// gemm_tiles.hip; many: gemm_group.h), the copy of misaligned operands, and
// the element-wise kernels around them (C = beta C, seeded fills, copies).
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <stdint.h>

#include "../hiplayer.h"
#include "blasx_ext.h"
#include "gemm_common.h"

namespace {

template <typename E>
__global__ void k_scale(int m, int n, E beta, int beta_zero, int tri, E *C, int64_t ldc)
{
    const int64_t total = (int64_t)m * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i % m, c = i / m;
        if (!tri_keep(tri, (int)r, (int)c)) continue;
        E *p = C + r + c * ldc;
        *p = beta_zero ? E(0) : beta * *p;
    }
}

__global__ void k_scale_z(int m, int n, double br, double bi, int beta_zero, int tri, cplx *C,
                          int64_t ldc)
{
    const int64_t total = (int64_t)m * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i % m, c = i / m;
        if (!tri_keep(tri, (int)r, (int)c)) continue;
        cplx *p = C + r + c * ldc;
        if (beta_zero) {
            *p = cplx{0.0, 0.0};
        } else {
            const cplx v = *p;
            *p = cplx{br * v.re - bi * v.im, br * v.im + bi * v.re};
        }
        if ((tri & BX_TRI_HERM) && r == c) p->im = 0.0;
    }
}

// SplitMix64 (Steele, Lea, Flood 2014); the host generator in fill.c is the same function
__device__ __forceinline__ uint64_t splitmix64(uint64_t x)
{
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double u11(uint64_t key)
{
    return ((double)(splitmix64(key) >> 11) * 0x1.0p-53) * 2.0 - 1.0;
}

__global__ void k_fill(int dtype, void *p, int64_t rows, int64_t cols, int64_t ld, uint64_t seed,
                       uint32_t id)
{
    const int64_t total = rows * cols;
    const uint64_t base = seed ^ ((uint64_t)id << 56);
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i % rows, c = i / rows;
        const int64_t o = r + c * ld;
        const uint64_t e = (uint64_t)i;
        if (dtype == BLASX_D) {
            ((double *)p)[o] = u11(base ^ e);
        } else if (dtype == BLASX_S) {
            ((float *)p)[o] = (float)u11(base ^ e);
        } else {
            ((double *)p)[2 * o] = u11(base ^ (2 * e));
            ((double *)p)[2 * o + 1] = u11(base ^ (2 * e + 1));
        }
    }
}

// plain streaming copy (16-byte vectors); also the reference kernel for
// calibrating HBM byte counters
__global__ void k_copy16(const int4 *__restrict__ src, int4 *__restrict__ dst, int64_t n16)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n16;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

thread_local char g_err[256];

int fail(const char *what, hipError_t e)
{
    snprintf(g_err, sizeof g_err, "%s: %s", what, hipGetErrorString(e));
    return BLASX_EHIP;
}

// ---- misaligned DGEMM operands ----
// An operand whose base or leading dimension is not 16-byte aligned is moved
// through registers by the tile kernels (64 TFLOP/s at 3001^3, where aligned
// operands reach 70).  A product large enough to pay for it copies the
// operand into an aligned workspace first (one HBM pass, leading dimension
// rounded up to 8 doubles).

__global__ void k_repack(const double *__restrict__ src, int64_t lds, double *__restrict__ dst,
                         int64_t ldd, int64_t rows, int64_t cols)
{
    for (int64_t c = blockIdx.y; c < cols; c += gridDim.y)
        for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < rows;
             r += (int64_t)gridDim.x * blockDim.x)
            dst[r + c * ldd] = src[r + c * lds];
}

void launch_repack(const double *src, int64_t lds, double *dst, int64_t ldd, int64_t rows,
                   int64_t cols, hipStream_t st)
{
    const int gx = (int)((rows + 255) / 256 < 16 ? (rows + 255) / 256 : 16);
    const int gy = (int)(cols < 8192 ? cols : 8192);
    hipLaunchKernelGGL(k_repack, dim3(gx, gy), dim3(256), 0, st, src, lds, dst, ldd, rows, cols);
}

// A device workspace reused across calls: a call's copies wait for the
// previous call's kernels (event on the device), growth waits on the host.
struct Workspace {
    void *p = nullptr;
    size_t cap = 0;
    hipEvent_t done = nullptr;
};
Workspace g_rws;
pthread_mutex_t g_rws_lock = PTHREAD_MUTEX_INITIALIZER;

// rows x cols of the stored operand behind op(A) (m x k) / op(B) (k x n)
inline void stored_dims(int op, int64_t r, int64_t c, int64_t &rows, int64_t &cols)
{
    rows = op ? c : r;
    cols = op ? r : c;
}

// 1: ran; 0: not taken (the caller runs the product on the operands as they
// are); <0: error
int dgemm_repacked(int ta, int tb, const bxh_problem_t &P, const bxh_seg_t &S, hipStream_t st)
{
    if (P.m < 128 || P.n < 128 || S.k < 16) return 0;
    const bool okA = aligned16(S.A, S.lda, 8), okB = aligned16(S.B, S.ldb, 8);
    if (okA && okB) return 0;
    // a copy of A costs ~16 MK bytes against 2 MNK flops: worth it from N ~ 4096
    if ((!okA && P.n < 4096) || (!okB && P.m < 4096)) return 0;
    int64_t ra, ca, rb, cb;
    stored_dims(ta, P.m, S.k, ra, ca);
    stored_dims(tb, S.k, P.n, rb, cb);
    const int64_t lda2 = (ra + 7) & ~(int64_t)7, ldb2 = (rb + 7) & ~(int64_t)7;
    const size_t bytesA = okA ? 0 : (size_t)lda2 * ca * 8, bytesB = okB ? 0 : (size_t)ldb2 * cb * 8;
    bxh_seg_t S2 = S;
    pthread_mutex_lock(&g_rws_lock);
    hipError_t e = hipSuccess;
    if (!g_rws.done) e = hipEventCreateWithFlags(&g_rws.done, hipEventDisableTiming);
    if (e == hipSuccess && bytesA + bytesB > g_rws.cap) {
        e = hipEventSynchronize(g_rws.done);
        if (e == hipSuccess && g_rws.p) e = hipFree(g_rws.p);
        g_rws.p = nullptr;
        g_rws.cap = 0;
        if (e == hipSuccess) e = hipMalloc(&g_rws.p, bytesA + bytesB);
        if (e == hipSuccess) g_rws.cap = bytesA + bytesB;
    }
    if (e == hipSuccess) e = hipStreamWaitEvent(st, g_rws.done, 0);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        pthread_mutex_unlock(&g_rws_lock);
        return fail("dgemm workspace", e);
    }
    double *wa = (double *)g_rws.p, *wb = (double *)((char *)g_rws.p + bytesA);
    if (!okA) {
        launch_repack((const double *)S.A, S.lda, wa, lda2, ra, ca, st);
        S2.A = wa;
        S2.lda = lda2;
    }
    if (!okB) {
        launch_repack((const double *)S.B, S.ldb, wb, ldb2, rb, cb, st);
        S2.B = wb;
        S2.ldb = ldb2;
    }
    int rc = bxh_gemm_tile(BLASX_D, &P, &S2, st);
    e = hipEventRecord(g_rws.done, st);
    pthread_mutex_unlock(&g_rws_lock);
    if (!rc && e != hipSuccess) rc = fail("dgemm workspace event", e);
    return rc ? rc : 1;
}

} // namespace

extern "C" {

const char *bxh_kernel_error(void) { return g_err; }

// the outcome of the kernel launch before it
int bx_launch_status(const char *what)
{
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(what, e);
}

void bxh_tile_dims(int dtype, int shape, int *bm, int *bn)
{
    switch (shape) {
    case BXH_SHAPE_32x32: *bm = *bn = 32; return;
    case BXH_SHAPE_64x64: *bm = *bn = 64; return;
    case BXH_SHAPE_128x64: *bm = 128, *bn = 64; return;
    default: *bm = bxh_tile_m(dtype), *bn = bxh_tile_n(dtype);
    }
}

int bxh_tile_m(int dtype)
{
    return dtype == BLASX_S ? Cfg<float>::BM : dtype == BLASX_D ? Cfg<double>::BM : Cfg<cplx>::BM;
}

int bxh_tile_n(int dtype)
{
    return dtype == BLASX_S ? Cfg<float>::BN : dtype == BLASX_D ? Cfg<double>::BN : Cfg<cplx>::BN;
}

int bx_launch_group_s(const bxh_problem_t *, int, const bxh_seg_t *, int, int, const int *, void *);
int bx_launch_group_d(const bxh_problem_t *, int, const bxh_seg_t *, int, int, const int *, void *);
int bx_launch_group_z(const bxh_problem_t *, int, const bxh_seg_t *, int, int, const int *, void *);

int bxh_gemm(int dtype, int opa, int opb, int m, int n, int k, const double *alpha,
             const void *A, int64_t lda, const void *B, int64_t ldb, const double *beta, void *C,
             int64_t ldc, void *stream)
{
    if (m <= 0 || n <= 0) return 0;
    if (opa < 0 || opa > 2 || opb < 0 || opb > 2 || k < 0) return BLASX_EINVAL;
    bxh_problem_t P;
    P.C = C;
    P.ldc = ldc;
    P.m = m;
    P.n = n;
    P.nseg = 1;
    P.seg_off = 0;
    P.opa = opa;
    P.opb = opb;
    P.tiles_m = (m + bxh_tile_m(dtype) - 1) / bxh_tile_m(dtype);
    P.tiles_n = (n + bxh_tile_n(dtype) - 1) / bxh_tile_n(dtype);
    P.tile_start = 0;
    P.alpha_re = alpha[0];
    P.alpha_im = dtype == BLASX_Z ? alpha[1] : 0.0;
    P.beta_re = beta[0];
    P.beta_im = dtype == BLASX_Z ? beta[1] : 0.0;
    P.beta_zero = (P.beta_re == 0.0 && P.beta_im == 0.0);
    P.tri = 0;
    P.tri_off = 0;
    P.shape = BXH_SHAPE_128x128;
    P.form = 0; /* set per operand alignment (bxh_gemm_tile) */
    bxh_seg_t S;
    S.A = A;
    S.B = B;
    S.lda = lda;
    S.ldb = ldb;
    S.k = k;
    hipStream_t st = (hipStream_t)stream;
    if (dtype != BLASX_S && dtype != BLASX_D && dtype != BLASX_Z) return BLASX_EINVAL;
    if (dtype == BLASX_D) {
        const int r = dgemm_repacked(opa != 0, opb != 0, P, S, st);
        if (r) return r < 0 ? r : 0;
    }
    return bxh_gemm_tile(dtype, &P, &S, st);
}

static int launch_grouped(int dtype, const bxh_problem_t *probs, int nprob, const bxh_seg_t *segs,
                          int total, int grid, const int *counts, void *stream)
{
    switch (dtype) {
    case BLASX_S: return bx_launch_group_s(probs, nprob, segs, total, grid, counts, stream);
    case BLASX_D: return bx_launch_group_d(probs, nprob, segs, total, grid, counts, stream);
    case BLASX_Z: return bx_launch_group_z(probs, nprob, segs, total, grid, counts, stream);
    }
    return BLASX_EINVAL;
}

int bxh_gemm_grouped(int dtype, const bxh_problem_t *probs_dev, int nprob,
                     const bxh_seg_t *segs_dev, int total_tiles, int grid, void *stream)
{
    if (nprob <= 0 || total_tiles <= 0) return 0;
    return launch_grouped(dtype, probs_dev, nprob, segs_dev, total_tiles, grid, nullptr, stream);
}

int bxh_gemm_grouped_dyn(int dtype, const bxh_problem_t *probs_dev, const bxh_seg_t *segs_dev,
                         const int *counts_dev, int grid, void *stream)
{
    if (grid <= 0) return BLASX_EINVAL;
    return launch_grouped(dtype, probs_dev, 0, segs_dev, 0, grid, counts_dev, stream);
}

int bxh_scale(int dtype, int m, int n, const double *beta, void *C, int64_t ldc, void *stream)
{
    return bxh_scale_tri(dtype, m, n, 0, beta, C, ldc, stream);
}

int bxh_scale_tri(int dtype, int m, int n, int tri, const double *beta, void *C, int64_t ldc,
                  void *stream)
{
    if (m <= 0 || n <= 0) return 0;
    const int64_t total = (int64_t)m * n;
    int grid = (int)((total + 255) / 256);
    if (grid > 65536) grid = 65536;
    hipStream_t st = (hipStream_t)stream;
    const int bz = (beta[0] == 0.0 && (dtype != BLASX_Z || beta[1] == 0.0));
    switch (dtype) {
    case BLASX_D:
        hipLaunchKernelGGL(k_scale<double>, dim3(grid), dim3(256), 0, st, m, n, beta[0], bz, tri,
                           (double *)C, ldc);
        break;
    case BLASX_S:
        hipLaunchKernelGGL(k_scale<float>, dim3(grid), dim3(256), 0, st, m, n, (float)beta[0], bz,
                           tri, (float *)C, ldc);
        break;
    case BLASX_Z:
        hipLaunchKernelGGL(k_scale_z, dim3(grid), dim3(256), 0, st, m, n, beta[0], beta[1], bz,
                           tri, (cplx *)C, ldc);
        break;
    default: return BLASX_EINVAL;
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("scale launch", e);
}

int bxh_copy_kernel(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return 0;
    if ((bytes & 15) || (((uintptr_t)dst | (uintptr_t)src) & 15)) return BLASX_EINVAL;
    const int64_t n16 = (int64_t)(bytes / 16);
    int64_t grid = (n16 + 255) / 256;
    if (grid > 65536) grid = 65536;
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream,
                       (const int4 *)src, (int4 *)dst, n16);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("copy launch", e);
}

int bxh_fill_uniform(int dtype, void *p, int64_t rows, int64_t cols, int64_t ld, uint64_t seed,
                     uint32_t id, void *stream)
{
    if (rows <= 0 || cols <= 0) return 0;
    if (dtype != BLASX_S && dtype != BLASX_D && dtype != BLASX_Z) return BLASX_EINVAL;
    const int64_t total = rows * cols;
    int grid = (int)((total + 255) / 256);
    if (grid > 262144) grid = 262144;
    hipLaunchKernelGGL(k_fill, dim3(grid), dim3(256), 0, (hipStream_t)stream, dtype, p, rows, cols,
                       ld, seed, id);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail("fill launch", e);
}

} // extern "C"
