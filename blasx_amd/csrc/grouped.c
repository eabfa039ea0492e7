/*
 * grouped.c -- grouped GEMM: many uneven GEMMs (mixed shapes, transposes
 * and element types) in one launch per element type.  No counterpart in the
 * reference, which issues one cublas call per tile product
 * (blas/blasx_dgemm.c:87-94).
 *
 * Descriptors are turned into a device-resident table of bxh_problem_t
 * (one block-tile range each) and bxh_seg_t (one K segment each) consumed
 * by the grouped kernel: a block finds its problem by its tile number (a graph
 * replay's blocks walk the tiles with a grid stride), the problems of the longest
 * K first, so a 64^3 request and an 8192^3 request share a launch.
 */
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

#include "internal.h"
#include "tilecost.h"

static int op_of(int dt, int t)
{
    if (t == 111) return BX_OP_N;
    if (t == 112) return BX_OP_T;
    if (t == 113) return dt == BLASX_Z ? BX_OP_C : BX_OP_T;
    return -1;
}

int bx_desc_check(const blasx_gemm_desc_t *d)
{
    if (d->dtype != BLASX_S && d->dtype != BLASX_D && d->dtype != BLASX_Z) return BLASX_EINVAL;
    const int opa = op_of(d->dtype, d->transa), opb = op_of(d->dtype, d->transb);
    if (opa < 0 || opb < 0 || d->M < 0 || d->N < 0 || d->K < 0) return BLASX_EINVAL;
    const int64_t nrowa = opa == BX_OP_N ? d->M : d->K, nrowb = opb == BX_OP_N ? d->K : d->N;
    if (d->lda < (nrowa > 1 ? nrowa : 1) || d->ldb < (nrowb > 1 ? nrowb : 1) ||
        d->ldc < (d->M > 1 ? d->M : 1))
        return BLASX_EINVAL;
    return 0;
}

static int desc_runs(const blasx_gemm_desc_t *x, int dtype)
{
    if (x->dtype != dtype || x->M == 0 || x->N == 0) return 0;
    const int az = x->alpha[0] == 0.0 && (dtype != BLASX_Z || x->alpha[1] == 0.0);
    return x->K != 0 && !az;
}

/* exchange two table entries (each problem has one segment) */
static void swap_entries(bxh_problem_t *probs, bxh_seg_t *segs, int i, int j)
{
    const bxh_problem_t p = probs[i];
    const bxh_seg_t s = segs[i];
    probs[i] = probs[j];
    segs[i] = segs[j];
    probs[j] = p;
    segs[j] = s;
}

/* restore the heap (least K at the root) of n entries below entry r */
static void sift(bxh_problem_t *probs, bxh_seg_t *segs, int r, int n)
{
    for (int c; (c = 2 * r + 1) < n; r = c) {
        if (c + 1 < n && segs[c + 1].k < segs[c].k) ++c;
        if (segs[r].k <= segs[c].k) return;
        swap_entries(probs, segs, r, c);
    }
}

/* Longest tiles first, so that the short ones fill the last wave: descending
 * K, by heap sort (in place: this path may not allocate).  Equal problems,
 * the usual launch, are left as they are. */
static void sort_by_k(bxh_problem_t *probs, bxh_seg_t *segs, int n)
{
    int sorted = 1;
    for (int i = 1; i < n && sorted; ++i) sorted = segs[i - 1].k >= segs[i].k;
    if (sorted) return;
    for (int r = n / 2 - 1; r >= 0; --r) sift(probs, segs, r, n);
    for (int end = n - 1; end > 0; --end) {
        swap_entries(probs, segs, 0, end);
        sift(probs, segs, 0, end);
    }
}

/* 64x64 tiles or 32x32 ones for the n problems of one launch: whichever
 * spreads over the CUs in less time, the tiles' total over 256 CUs plus half
 * the longest (what longest-first order leaves uneven), tilecost.h */
static int small_shape(int dtype, const bxh_problem_t *probs, const bxh_seg_t *segs, int n)
{
    double t[2];
    const int s[2] = {BXC_64x64, BXC_32x32};
    for (int j = 0; j < 2; ++j) {
        double sum = 0, most = 0;
        for (int i = 0; i < n; ++i) {
            const bx_cost_t *c = probs[i].form == BXH_FORM_DMA ? &BX_COST_DMA[dtype][s[j]]
                                                               : &BX_COST_REG[dtype][s[j]];
            const double one = bx_cost_tile(c, segs[i].k);
            sum += one * (double)bx_cost_tiles(s[j], probs[i].m, probs[i].n);
            if (one > most) most = one;
        }
        t[j] = sum / 256 + 0.5 * most;
    }
    return t[1] < t[0] ? BXH_SHAPE_32x32 : BXH_SHAPE_64x64;
}

/* tile counts and starts of problems [first, first + n), from 0 */
static int place_tiles(int dtype, bxh_problem_t *probs, int n)
{
    int total = 0;
    for (int i = 0; i < n; ++i) {
        int bm, bn;
        bxh_tile_dims(dtype, probs[i].shape, &bm, &bn);
        probs[i].tiles_m = (probs[i].m + bm - 1) / bm;
        probs[i].tiles_n = (probs[i].n + bn - 1) / bn;
        probs[i].tile_start = total;
        total += probs[i].tiles_m * probs[i].tiles_n;
    }
    return total;
}

/* A complex problem's shape in a launch of `load` 128x64 tiles of its type:
 * 128x64 where they take one round of two tiles on each of 256 CUs, while 64x64
 * tiles, three on a CU, would begin a second, uneven one (one 2048^3 934 against
 * 1134 us, four of 1024^3 478 against 521, 256 of 128^3 92 against 105), and no
 * half of a tile stays empty.  With fewer tiles 64x64 or 32x32 spread better (8
 * of 512^3: 130 against 138 us); with more the two are level on whole tiles (four
 * of 4096^3 28.6 ms) and 64x64 ahead on ragged ones (12 of 450x1100x900 721
 * against 842 us, 24 of 300x3000x700 1844 against 2252), until K is so long that
 * the smaller tiles miss L2 (64 of 256x16384x8192 230 against 242 ms, two of 8192^3
 * 114.8 against 117.0, 32 of 256x8192x4096 28.8 against 29.4). */
static int complex_shape(int M, int K, int64_t load)
{
    const int over = (M + 127) / 128 * 128 - (M + 63) / 64 * 64;
    const int one_round = load > 384 && load <= 512, long_k = load >= 2048 && K >= 4096;
    return (one_round || long_k) && 16 * over <= M ? BXH_SHAPE_128x64 : BXH_SHAPE_64x64;
}

/* Fill problem/segment tables for the descriptors of one dtype (device
 * pointers in the descriptors).  Descriptors with alpha == 0 or K == 0 are
 * skipped (the caller scales C separately).  A real problem's shape comes from
 * bx_grouped_shape, a complex one's from complex_shape, given the launch's
 * load: its tile count at the large tile; problems on 64x64 tiles and those
 * whose operands do not take the DMA share one choice of 64x64 or 32x32.  The first nprob[0]
 * problems (total[0] tiles) are those, the next nprob[1] (total[1] tiles, a
 * launch of their own) the 128-row shapes; big = 0 puts all in the first. */
void bx_grouped_fill(const blasx_gemm_desc_t *d, int n, int dtype, bxh_problem_t *probs,
                     bxh_seg_t *segs, int big, int nprob[2], int total[2])
{
    const int bm0 = bxh_tile_m(dtype), bn0 = bxh_tile_n(dtype);
    int64_t load = 0;
    for (int i = 0; i < n; ++i)
        if (desc_runs(&d[i], dtype))
            load += (int64_t)((d[i].M + bm0 - 1) / bm0) * ((d[i].N + bn0 - 1) / bn0);
    int np = 0, nbig = 0;
    /* the previous problem's choice, reused while M, N and K repeat: the
     * table lookup takes a lock and interpolates, which on launches of many
     * small equal problems cost more host time than the kernel took */
    int lm = -1, ln = -1, lk = -1, shape = 0;
    for (int i = 0; i < n; ++i) {
        const blasx_gemm_desc_t *x = &d[i];
        if (!desc_runs(x, dtype)) continue;
        bxh_problem_t *P = &probs[np];
        if (x->M != lm || x->N != ln || x->K != lk) {
            shape = dtype == BLASX_Z ? complex_shape(x->M, x->K, load)
                                     : bx_grouped_shape(dtype, x->M, x->N, x->K, load);
            lm = x->M;
            ln = x->N;
            lk = x->K;
        }
        memset(P, 0, sizeof *P);
        P->C = x->C;
        P->ldc = x->ldc;
        P->m = x->M;
        P->n = x->N;
        P->nseg = 1;
        P->opa = op_of(dtype, x->transa);
        P->opb = op_of(dtype, x->transb);
        P->alpha_re = x->alpha[0];
        P->alpha_im = dtype == BLASX_Z ? x->alpha[1] : 0.0;
        P->beta_re = x->beta[0];
        P->beta_im = dtype == BLASX_Z ? x->beta[1] : 0.0;
        P->beta_zero = P->beta_re == 0.0 && P->beta_im == 0.0;
        segs[np].A = x->A;
        segs[np].B = x->B;
        segs[np].lda = x->lda;
        segs[np].ldb = x->ldb;
        segs[np].k = x->K;
        P->form = bxh_tile_form(dtype, P->opa, P->opb, P->m, P->n, &segs[np]);
        P->shape = big && P->form == BXH_FORM_DMA ? shape : BXH_SHAPE_64x64;
        /* small problems stay in front of the big ones */
        if (P->shape != BXH_SHAPE_64x64)
            ++nbig;
        else if (nbig)
            swap_entries(probs, segs, np, np - nbig);
        ++np;
    }
    const int ns = np - nbig;
    if (ns) {
        const int s = small_shape(dtype, probs, segs, ns);
        for (int i = 0; i < ns; ++i) probs[i].shape = s;
    }
    sort_by_k(probs, segs, ns);
    sort_by_k(probs + ns, segs + ns, nbig);
    for (int i = 0; i < np; ++i) probs[i].seg_off = i;
    nprob[0] = ns;
    nprob[1] = nbig;
    total[0] = place_tiles(dtype, probs, ns);
    total[1] = place_tiles(dtype, probs + ns, nbig);
}

/* the launches of one dtype's tables */
static int launch_tables(int dtype, const bxh_problem_t *probs, const bxh_seg_t *segs,
                         const int nprob[2], const int total[2], void *st, int *launches)
{
    int rc = 0;
    if (nprob[0]) {
        rc = bxh_gemm_grouped(dtype, probs, nprob[0], segs, total[0], 0, st);
        ++*launches;
    }
    if (!rc && nprob[1]) {
        rc = bxh_gemm_grouped(dtype, probs + nprob[0], nprob[1], segs, total[1], BXH_GROUP_BIG, st);
        ++*launches;
    }
    return rc;
}

static double desc_flops(const blasx_gemm_desc_t *d, int n, int dtype)
{
    double f = 0;
    for (int i = 0; i < n; ++i)
        if (d[i].dtype == dtype)
            f += (dtype == BLASX_Z ? 8.0 : 2.0) * d[i].M * (double)d[i].N * d[i].K;
    return f;
}

/* ---- blasx_gemm_grouped_device ---- */
/* table staging: the host runs up to GRING calls ahead of the GPU */
enum { GRING = 4 };
static pthread_mutex_t g_glock = PTHREAD_MUTEX_INITIALIZER;
static struct {
    void *host, *dev, *done;
    size_t cap;
} g_gring[GRING];
static unsigned g_gnext;

BX_EXPORT int blasx_gemm_grouped_device(const blasx_gemm_desc_t *d, int n, void *stream)
{
    if (bx_ensure_init() != 0) return BLASX_ENOGPU;
    if (n < 0 || (n > 0 && !d)) return BLASX_EINVAL;
    for (int i = 0; i < n; ++i)
        if (bx_desc_check(&d[i])) return BLASX_EINVAL;
    void *st = stream ? stream : g_bx.s_comp;
    int rc = 0;
    /* degenerate descriptors: C = beta C */
    for (int i = 0; i < n && !rc; ++i) {
        const int az = d[i].alpha[0] == 0.0 && (d[i].dtype != BLASX_Z || d[i].alpha[1] == 0.0);
        if (d[i].M > 0 && d[i].N > 0 && (d[i].K == 0 || az))
            rc = bxh_scale(d[i].dtype, d[i].M, d[i].N, d[i].beta, d[i].C, d[i].ldc, st);
    }
    if (rc || n == 0) return rc;

    /* one table entry per descriptor, whatever its type: problems, then segments */
    const size_t seg_at = (size_t)n * sizeof(bxh_problem_t);
    const size_t need = seg_at + (size_t)n * sizeof(bxh_seg_t);
    pthread_mutex_lock(&g_glock);
    const unsigned slot = g_gnext++ % GRING;
    if (!g_gring[slot].done) rc = bxh_event_create(&g_gring[slot].done, 0);
    if (!rc) rc = bxh_event_sync(g_gring[slot].done); /* this slot's tables are consumed */
    if (!rc && need > g_gring[slot].cap) {
        bxh_host_free(g_gring[slot].host);
        bxh_free(g_gring[slot].dev);
        g_gring[slot].host = g_gring[slot].dev = NULL;
        g_gring[slot].cap = 0;
        rc = bxh_host_malloc(&g_gring[slot].host, need);
        if (!rc) rc = bxh_malloc(&g_gring[slot].dev, need);
        if (!rc) g_gring[slot].cap = need;
    }
    const int dts[3] = {BLASX_S, BLASX_D, BLASX_Z};
    int np[3][2] = {{0}}, total[3][2] = {{0}}, first[3], used = 0, launches = 0;
    double flops = 0;
    if (!rc) {
        bxh_problem_t *probs = (bxh_problem_t *)g_gring[slot].host;
        bxh_seg_t *segs = (bxh_seg_t *)((char *)g_gring[slot].host + seg_at);
        for (int k = 0; k < 3; ++k) {
            first[k] = used;
            bx_grouped_fill(d, n, dts[k], probs + used, segs + used, 1, np[k], total[k]);
            const int runs = np[k][0] + np[k][1];
            used += runs;
            if (runs) flops += desc_flops(d, n, dts[k]);
        }
        if (used) rc = bxh_memcpy_h2d_async(g_gring[slot].dev, g_gring[slot].host, need, st);
    }
    for (int k = 0; k < 3 && !rc; ++k)
        rc = launch_tables(dts[k], (const bxh_problem_t *)g_gring[slot].dev + first[k],
                           (const bxh_seg_t *)((char *)g_gring[slot].dev + seg_at) + first[k], np[k],
                           total[k], st, &launches);
    if (g_gring[slot].done) {
        const int re = bxh_event_record(g_gring[slot].done, st);
        if (!rc) rc = re;
    }
    pthread_mutex_unlock(&g_glock);
    if (!rc) {
        BX_STAT_ADD(kernel_launches, launches);
        bx_stat_flops(flops);
    }
    return rc;
}

/* ---- blasx_gemm_grouped_device_noalloc ----
 * The same launches as blasx_gemm_grouped_device with the problem and
 * segment tables in the static per-GPU table store of hip/noalloc.hip
 * instead of a device buffer the library allocates: no hipMalloc, hipFree or
 * other allocating call on this path.  The host side builds the tables in a
 * static (pageable) host buffer and copies them on `stream`.  Calls are
 * ordered on the device: a call's table copy waits for the event the
 * previous call recorded after its kernels, on whatever stream that ran, so
 * the store is never overwritten under a running launch.  The store keeps the
 * last call's tables; nothing in it needs to start at zero. */
static pthread_mutex_t g_nalock = PTHREAD_MUTEX_INITIALIZER;
static unsigned char g_na_host[BXH_NOALLOC_SCRATCH_BYTES] __attribute__((aligned(256)));
static void *g_na_copied; /* recorded after the host tables were last copied */

BX_EXPORT int blasx_gemm_grouped_device_noalloc(const blasx_gemm_desc_t *d, int n, void *stream)
{
    if (bx_ensure_init() != 0) return BLASX_ENOGPU;
    if (n < 0 || (n > 0 && !d)) return BLASX_EINVAL;
    if (n > BXH_NOALLOC_MAX_PROBLEMS) {
        bx_log(0, "blasx_gemm_grouped_device_noalloc: %d problems exceed the static table of "
                  "%d (use blasx_gemm_grouped_device)",
               n, BXH_NOALLOC_MAX_PROBLEMS);
        return BLASX_ERANGE;
    }
    for (int i = 0; i < n; ++i)
        if (bx_desc_check(&d[i])) return BLASX_EINVAL;
    void *st = stream ? stream : g_bx.s_comp;
    pthread_mutex_lock(&g_nalock);
    void *store = NULL, *done = NULL;
    int rc = bxh_noalloc_scratch(&store, &done);
    if (rc) bx_log(0, "noalloc table store: %s", bxh_noalloc_error());
    if (!rc && !g_na_copied) rc = bxh_event_create(&g_na_copied, 0);
    /* the host tables are rewritten only after their last copy has read them */
    if (!rc) rc = bxh_event_sync(g_na_copied);
    /* and the device tables only after the previous call's kernels */
    if (!rc) rc = bxh_stream_wait_event(st, done);
    for (int i = 0; i < n && !rc; ++i) {
        const int az = d[i].alpha[0] == 0.0 && (d[i].dtype != BLASX_Z || d[i].alpha[1] == 0.0);
        if (d[i].M > 0 && d[i].N > 0 && (d[i].K == 0 || az))
            rc = bxh_scale(d[i].dtype, d[i].M, d[i].N, d[i].beta, d[i].C, d[i].ldc, st);
    }
    const int dts[3] = {BLASX_S, BLASX_D, BLASX_Z};
    int launches = 0;
    double flops = 0;
    for (int k = 0; k < 3 && !rc && n > 0; ++k) {
        unsigned char *h = g_na_host + (size_t)k * BXH_NOALLOC_SLOT_BYTES;
        char *dv = (char *)store + (size_t)k * BXH_NOALLOC_SLOT_BYTES;
        bxh_problem_t *probs = (bxh_problem_t *)h;
        bxh_seg_t *segs = (bxh_seg_t *)(h + BXH_NOALLOC_SEG_OFFSET);
        int nprob[2], total[2];
        bx_grouped_fill(d, n, dts[k], probs, segs, 1, nprob, total);
        const size_t np = (size_t)(nprob[0] + nprob[1]);
        if (np == 0) continue;
        rc = bxh_memcpy_h2d_async(dv, h, np * sizeof(bxh_problem_t), st);
        if (!rc)
            rc = bxh_memcpy_h2d_async(dv + BXH_NOALLOC_SEG_OFFSET, h + BXH_NOALLOC_SEG_OFFSET,
                                      np * sizeof(bxh_seg_t), st);
        if (!rc)
            rc = launch_tables(dts[k], (const bxh_problem_t *)dv,
                               (const bxh_seg_t *)(dv + BXH_NOALLOC_SEG_OFFSET), nprob, total, st,
                               &launches);
        flops += desc_flops(d, n, dts[k]);
    }
    if (!rc) rc = bxh_event_record(g_na_copied, st);
    if (!rc) rc = bxh_event_record(done, st);
    pthread_mutex_unlock(&g_nalock);
    if (!rc) {
        BX_STAT_ADD(kernel_launches, launches);
        bx_stat_flops(flops);
    }
    return rc;
}
