/*
 * syrk.c -- symmetric and Hermitian rank-k updates on the GPU:
 * cblas_{s,d,c,z}syrk, cblas_{c,z}herk and their f77 forms,
 *   C = alpha op(A) op(A)^T + beta C   (op(A)^H and real alpha, beta for HERK)
 * on the triangle Uplo names.
 *
 * Replaces blas/ssyrk.c:15-95, blas/dsyrk.c:15-95, blas/csyrk.c:15-95,
 * blas/zsyrk.c:15-95, blas/cherk.c:15-108 and blas/zherk.c:15-108, which validate and then always forward to the CPU
 * BLAS (blas/dsyrk.c:46-49: both dispatch branches choose the CPU).  Kept
 * from them: the validation order and info numbers (blas/dsyrk.c:33-38,
 * lowest number wins), the xerbla_ names, the "N or K above 1000" size test
 * the reference computes (blas/dsyrk.c:48; 500 for complex types).  The
 * GPU runs what the reference's unused triangular tile helpers describe
 * (blas/blasx_mem_control.c:3-22, 189-219): only the C tiles on the stored
 * triangle, the diagonal tiles masked.
 *
 * CSYRK and CHERK (complex64) run on the FP32 matrix cores as a full product
 * whose stored triangle is copied back (bx_gpu_crank, level3.c).  For the
 * other types, host operands go through the tile runtime (bx_tile_syrk) and
 * operands in HBM run as one launch here, over the tiles on the stored
 * triangle, those on the diagonal masked.
 *
 * Deviations (netlib semantics): RowMajor is computed (the other triangle
 * with the transposition flipped); ZSYRK rejects ConjTrans (info 2), as
 * netlib does; f77 argument errors report the lowest parameter number.
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "blasx.h"
#include "cpu_forward.h"
#include "internal.h"

/* ---------------------------------------------------------------- device */
/* operands, C and the launch on `stream` (NULL: the library's compute
 * stream); asynchronous, like the other device entry points.  With B (SYR2K)
 * C = alpha op(A) op(B)^T + alpha op(B) op(A)^T + beta C on the triangle. */
int bx_device_syrk(int dt, int tri, int opa, int N, int K, const double *alpha, const void *A,
                   int64_t lda, const void *B, int64_t ldb, const double *beta, void *C,
                   int64_t ldc, void *stream)
{
    return bx_device_syr2k(dt, tri, opa, N, K, alpha, A, lda, B, ldb, B, ldb, beta, C, ldc,
                           stream);
}

/* the same with the second term's op(B) rows taken from B2 (HER2K passes a
 * copy of B scaled so that one alpha serves both terms) */
int bx_device_syr2k(int dt, int tri, int opa, int N, int K, const double *alpha, const void *A,
                    int64_t lda, const void *B, int64_t ldb, const void *B2, int64_t ldb2,
                    const double *beta, void *C, int64_t ldc, void *stream)
{
    if (bx_ensure_init() != 0) return BLASX_ENOGPU;
    void *st = stream ? stream : g_bx.s_comp;
    if (N <= 0) return 0;
    if (K == 0 || (alpha[0] == 0.0 && alpha[1] == 0.0))
        return bxh_scale_tri(dt, N, N, tri, beta, C, ldc, st);

    /* one launch over the tiles on the stored triangle; term 1: op(A) x op(B)^T
     * (op(A)^T for SYRK), term 2 (SYR2K): op(B2) x op(A)^T */
    bxh_problem_t P;
    memset(&P, 0, sizeof P);
    P.C = C;
    P.ldc = ldc;
    P.m = P.n = N;
    P.nseg = B ? 2 : 1;
    P.opa = opa;
    P.opb = opa != BX_OP_N ? BX_OP_N : (tri & BX_TRI_HERM) ? BX_OP_C : BX_OP_T;
    P.alpha_re = alpha[0];
    P.alpha_im = alpha[1];
    P.beta_re = beta[0];
    P.beta_im = beta[1];
    P.beta_zero = beta[0] == 0.0 && beta[1] == 0.0;
    P.tri = tri;
    const bxh_seg_t S[2] = {{A, B ? B : A, lda, B ? ldb : lda, K},
                            {B2 ? B2 : B, A, B2 ? ldb2 : ldb, lda, K}};
    const int rc = bxh_gemm_tile(dt, &P, S, st);
    if (!rc) {
        BX_STAT_ADD(kernel_launches, 1);
        bx_stat_flops(P.nseg * (dt == BLASX_Z ? 4.0 : 1.0) * (double)N * (N + 1) * K);
    }
    return rc;
}

/* ------------------------------------------------------------------ ABI */
static const char *syrk_name(int dt, int herk)
{
    if (herk) return dt == BLASX_C ? "CHERK" : "ZHERK"; /* blas/zherk.c:13, blas/cherk.c:13 */
    return dt == BLASX_S ? "SSYRK " : dt == BLASX_D ? "DSYRK " : dt == BLASX_C ? "CSYRK " : "ZSYRK ";
}

static int trans_ok(int dt, int herk, int t)
{
    if (t == CblasNoTrans) return 1;
    if (herk) return t == CblasConjTrans;
    if (dt == BLASX_Z || dt == BLASX_C) return t == CblasTrans;
    return t == CblasTrans || t == CblasConjTrans; /* C means T for real data */
}

static void scalar2(int dt, int herk, const void *v, double out[2])
{
    if (dt == BLASX_S || (dt == BLASX_C && herk)) {
        out[0] = *(const float *)v, out[1] = 0;
    } else if (dt == BLASX_C) {
        out[0] = ((const float *)v)[0], out[1] = ((const float *)v)[1];
    } else if (dt == BLASX_D || herk) {
        out[0] = *(const double *)v, out[1] = 0;
    } else {
        out[0] = ((const double *)v)[0], out[1] = ((const double *)v)[1];
    }
}

/* the CPU BLAS's own routine, Order passed through, as the reference does
 * (blas/dsyrk.c:58) */
static int cpu_syrk(int dt, int herk, int order, int uplo, int trans, int N, int K,
                    const void *alpha, const void *A, int lda, const void *beta, void *C, int ldc)
{
    if (bx_cpublas_load() != 0) return BLASX_ECPU;
    if (herk && dt == BLASX_C)
        bx_cpu_cherk(order, uplo, trans, N, K, *(const float *)alpha, A, lda,
                     *(const float *)beta, C, ldc);
    else if (herk)
        bx_cpu_zherk(order, uplo, trans, N, K, *(const double *)alpha, A, lda,
                     *(const double *)beta, C, ldc);
    else if (dt == BLASX_C)
        bx_cpu_csyrk(order, uplo, trans, N, K, alpha, A, lda, beta, C, ldc);
    else if (dt == BLASX_S)
        bx_cpu_ssyrk(order, uplo, trans, N, K, *(const float *)alpha, A, lda,
                     *(const float *)beta, C, ldc);
    else if (dt == BLASX_D)
        bx_cpu_dsyrk(order, uplo, trans, N, K, *(const double *)alpha, A, lda,
                     *(const double *)beta, C, ldc);
    else
        bx_cpu_zsyrk(order, uplo, trans, N, K, alpha, A, lda, beta, C, ldc);
    BX_STAT_ADD(calls_cpu, 1);
    return 0;
}

static void syrk_entry(int dt, int herk, int order, int Uplo, int Trans, int N, int K,
                       const void *alpha, const void *A, int lda, const void *beta, void *C,
                       int ldc)
{
    const char *name = syrk_name(dt, herk);
    int uplo = Uplo, trans = Trans, info = 0;
    if (order == CblasRowMajor) {
        /* a row-major C is the column-major C^T: the other triangle, with
         * op(A) and op(A)^T exchanged */
        uplo = Uplo == CblasUpper ? CblasLower : Uplo == CblasLower ? CblasUpper : Uplo;
        if (trans_ok(dt, herk, Trans))
            trans = Trans != CblasNoTrans ? CblasNoTrans : herk ? CblasConjTrans : CblasTrans;
    } else if (order != CblasColMajor) {
        xerbla_(name, &info); /* info 0: bad Order, as OpenBLAS reports it */
        return;
    }
    const int nrowa = trans == CblasNoTrans ? N : K;
    if (ldc < (N > 1 ? N : 1)) info = 10;
    if (lda < (nrowa > 1 ? nrowa : 1)) info = 7;
    if (K < 0) info = 4;
    if (N < 0) info = 3;
    if (!trans_ok(dt, herk, trans)) info = 2;
    if (uplo != CblasUpper && uplo != CblasLower) info = 1;
    if (info != 0) {
        xerbla_(name, &info);
        return;
    }
    if (N == 0) return;
    double al[2], be[2];
    scalar2(dt, herk, alpha, al);
    scalar2(dt, herk, beta, be);
    const int no_product = K == 0 || (al[0] == 0.0 && al[1] == 0.0);
    if (no_product && be[0] == 1.0 && be[1] == 0.0) return;

    bx_config();
    const int thr = (dt == BLASX_Z || dt == BLASX_C) ? g_bx.min_dim_cplx : g_bx.min_dim_real;
    if (!(N > thr || K > thr)) {
        if (cpu_syrk(dt, herk, order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc) != 0)
            bx_fatal("%s: no CPU BLAS could be loaded for a CPU-sized call (set BLASX_CPUBLAS)",
                     name);
        return;
    }
    const int tri = (uplo == CblasLower ? BX_TRI_LOWER : BX_TRI_UPPER) | (herk ? BX_TRI_HERM : 0);
    const int opa = trans == CblasNoTrans ? BX_OP_N : herk ? BX_OP_C : BX_OP_T;
    int rc = bx_ensure_init();
    if (rc == 0 && dt == BLASX_C) {
        /* complex64 on the FP32 matrix cores (level3.c) */
        rc = bx_gpu_crank(herk, uplo, trans, N, K, al, A, lda, NULL, 0, be, C, ldc);
        if (rc == BLASX_ENOMEM) {
            bx_log(1, "%s: operands do not fit in HBM; running on the CPU BLAS", name);
            if (cpu_syrk(dt, herk, order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc) != 0)
                bx_fatal("%s: no CPU BLAS could be loaded (set BLASX_CPUBLAS)", name);
            return;
        }
        if (rc == 0) {
            BX_STAT_ADD(calls_gpu, 1);
            return;
        }
    } else if (rc == 0) {
        if (bxh_pointer_is_pinned(C) == 2 && (no_product || bxh_pointer_is_pinned(A) == 2)) {
            /* operands already in HBM: run in place */
            rc = bx_device_syrk(dt, tri, opa, N, K, al, A, lda, NULL, 0, be, C, ldc, NULL);
            if (rc == 0) rc = bxh_stream_sync(g_bx.s_comp);
        } else if (no_product) {
            /* C = beta C on the triangle: host work, no product to run */
            if (cpu_syrk(dt, herk, order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc) != 0)
                bx_fatal("%s: no CPU BLAS could be loaded (set BLASX_CPUBLAS)", name);
            return;
        } else {
            rc = bx_tile_syrk(dt, tri, opa, N, K, al, A, lda, be, C, ldc);
        }
        if (rc == 0) {
            BX_STAT_ADD(calls_gpu, 1);
            return;
        }
    }
    if (bx_gpu_failed(name, rc, !bx_in_hbm(A) && !bx_in_hbm(C)) &&
        cpu_syrk(dt, herk, order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc) != 0)
        bx_fatal("%s: no CPU BLAS could be loaded for the fallback (set BLASX_CPUBLAS)", name);
}

BX_EXPORT void cblas_ssyrk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const float alpha, const float *A, const int lda, const float beta,
                           float *C, const int ldc)
{
    syrk_entry(BLASX_S, 0, Order, Uplo, Trans, N, K, &alpha, A, lda, &beta, C, ldc);
}

BX_EXPORT void cblas_dsyrk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const double alpha, const double *A, const int lda, const double beta,
                           double *C, const int ldc)
{
    syrk_entry(BLASX_D, 0, Order, Uplo, Trans, N, K, &alpha, A, lda, &beta, C, ldc);
}

BX_EXPORT void cblas_zsyrk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const void *alpha, const void *A, const int lda, const void *beta,
                           void *C, const int ldc)
{
    syrk_entry(BLASX_Z, 0, Order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc);
}

BX_EXPORT void cblas_zherk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const double alpha, const void *A, const int lda, const double beta,
                           void *C, const int ldc)
{
    syrk_entry(BLASX_Z, 1, Order, Uplo, Trans, N, K, &alpha, A, lda, &beta, C, ldc);
}

BX_EXPORT void cblas_csyrk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const void *alpha, const void *A, const int lda, const void *beta,
                           void *C, const int ldc)
{
    syrk_entry(BLASX_C, 0, Order, Uplo, Trans, N, K, alpha, A, lda, beta, C, ldc);
}

BX_EXPORT void cblas_cherk(const enum CBLAS_ORDER Order, const enum CBLAS_UPLO Uplo,
                           const enum CBLAS_TRANSPOSE Trans, const int N, const int K,
                           const float alpha, const void *A, const int lda, const float beta,
                           void *C, const int ldc)
{
    syrk_entry(BLASX_C, 1, Order, Uplo, Trans, N, K, &alpha, A, lda, &beta, C, ldc);
}

/* f77: info 1 for a bad UPLO, 2 for a bad TRANS character; both checks
 * run and the later one wins, so two bad characters report 2
 * (blas/dsyrk.c:83-85, blas/zherk.c:89-91), then the ColMajor CBLAS path */
static int f77_syrk_args(const char *name, const char *uplo, const char *trans, int *u, int *t)
{
    int info = 0;
    switch (*uplo) {
    case 'U': case 'u': *u = CblasUpper; break;
    case 'L': case 'l': *u = CblasLower; break;
    default: info = 1;
    }
    switch (*trans) {
    case 'N': case 'n': *t = CblasNoTrans; break;
    case 'T': case 't': *t = CblasTrans; break;
    case 'C': case 'c': *t = CblasConjTrans; break;
    default: info = 2;
    }
    if (info) xerbla_(name, &info);
    return info;
}

BX_EXPORT void ssyrk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const float *alpha, const float *A, const int *lda, const float *beta,
                      float *C, const int *ldc)
{
    int u, t;
    if (f77_syrk_args("SSYRK ", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_S, 0, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}

BX_EXPORT void dsyrk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const double *alpha, const double *A, const int *lda, const double *beta,
                      double *C, const int *ldc)
{
    int u, t;
    if (f77_syrk_args("DSYRK ", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_D, 0, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}

BX_EXPORT void zsyrk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const void *alpha, const void *A, const int *lda, const void *beta, void *C,
                      const int *ldc)
{
    int u, t;
    if (f77_syrk_args("ZSYRK ", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_Z, 0, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}

BX_EXPORT void zherk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const double *alpha, const void *A, const int *lda, const double *beta,
                      void *C, const int *ldc)
{
    int u, t;
    if (f77_syrk_args("ZHERK", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_Z, 1, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}

BX_EXPORT void csyrk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const void *alpha, const void *A, const int *lda, const void *beta, void *C,
                      const int *ldc)
{
    int u, t;
    if (f77_syrk_args("CSYRK ", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_C, 0, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}

BX_EXPORT void cherk_(const char *uplo, const char *trans, const int *n, const int *k,
                      const float *alpha, const void *A, const int *lda, const float *beta,
                      void *C, const int *ldc)
{
    int u, t;
    if (f77_syrk_args("CHERK", uplo, trans, &u, &t)) return;
    syrk_entry(BLASX_C, 1, CblasColMajor, u, t, *n, *k, alpha, A, *lda, beta, C, *ldc);
}
