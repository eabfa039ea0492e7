// level3.hip -- the non-GEMM kernels of the level-3 routines built on GEMMs:
//  * operand materialisation (SYMM, HEMM, TRMM, TRSM): the full symmetric or
//    Hermitian matrix from its stored triangle, or the triangular matrix with
//    the other triangle zero (and a unit diagonal when asked).  HBM-bound
//    element work: one pass over an n x n matrix, the mirrored half staged
//    through LDS in 32 x 32 tiles so both its reads and its writes coalesce;
//  * a tiled (conjugate) transpose (TRSM's op(A) and its Right side);
//  * TRSM's diagonal-block solve: substitution on 64-row blocks (32 for
//    complex), one column per thread.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../hiplayer.h"
#include "blasx_ext.h"

namespace {

// complex elements: T is double (complex128) or float (complex64)
template <typename T> struct cx {
    T re, im;
};
using z16 = cx<double>;
using c8 = cx<float>;

template <typename E> struct is_cx { static constexpr bool value = false; };
template <typename T> struct is_cx<cx<T>> { static constexpr bool value = true; };

template <typename E> __device__ __forceinline__ E conj_of(E v)
{
    if constexpr (is_cx<E>::value) return E{v.re, -v.im};
    else return v;
}
template <typename E> __device__ __forceinline__ E real_of(E v)
{
    if constexpr (is_cx<E>::value) return E{v.re, 0};
    else return v;
}
template <typename E> __device__ __forceinline__ E zero_of()
{
    if constexpr (is_cx<E>::value) return E{0, 0};
    else return E(0);
}
template <typename E> __device__ __forceinline__ E one_of()
{
    if constexpr (is_cx<E>::value) return E{1, 0};
    else return E(1);
}

// acc - a * b, and a / b, for the substitution
template <typename E> __device__ __forceinline__ E sub_mul(E acc, E a, E b)
{
    if constexpr (is_cx<E>::value)
        return E{acc.re - (a.re * b.re - a.im * b.im), acc.im - (a.re * b.im + a.im * b.re)};
    else return acc - a * b;
}
// c ? a : b by value, component by component (a conditional on two struct
// lvalues may select their addresses and pin a register array in memory)
template <typename E> __device__ __forceinline__ E pick(bool c, E a, E b)
{
    if constexpr (is_cx<E>::value) return E{c ? a.re : b.re, c ? a.im : b.im};
    else return c ? a : b;
}
// complex division by Smith's method (Smith 1962), which avoids overflow in
// |b|^2: with p the larger-magnitude part of b and o the other, r = o / p and
// d = p + o r; |b.re| >= |b.im| gives ((a.re + a.im r) + i (a.im - a.re r)) / d,
// else ((a.im + a.re r) + i (a.im r - a.re)) / d.  Written with selects, not
// branches, so unrolled callers stay one basic block.
template <typename E> __device__ __forceinline__ E divide(E a, E b)
{
    if constexpr (is_cx<E>::value) {
        const bool big = fabs(b.re) >= fabs(b.im);
        const auto p = big ? b.re : b.im, o = big ? b.im : b.re;
        const auto u = big ? a.re : a.im, v = big ? a.im : a.re;
        const auto r = o / p, d = p + o * r;
        const auto t = v - u * r;
        return E{(u + v * r) / d, (big ? t : -t) / d};
    } else {
        return a / b;
    }
}

constexpr int TB = 32;

// Block (bx, by) owns destination tile rows [by*32, +32), columns [bx*32, +32)
// of the n x n matrix A; 256 threads as 32 (row) x 8 (column step).  Tiles
// wholly inside the stored triangle exit at once (uniformly per block).
template <typename E>
__global__ __launch_bounds__(256) void k_tri_fill(int n, int lower, int mode, E *A, int64_t lda)
{
    __shared__ E tile[TB][TB + 1];
    const int bi = blockIdx.y, bj = blockIdx.x;
    if (lower ? bi > bj : bi < bj) return; // stored side, off the diagonal
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const bool mirror = mode == BX_FILL_SYM || mode == BX_FILL_HERM;
    if (mirror) {
        // the source of tile (bi, bj) is tile (bj, bi): tile[a][b] = A(bj*32 + a, bi*32 + b)
        for (int k = ty; k < TB; k += 8) {
            const int r = bj * TB + tx, c = bi * TB + k;
            if (r < n && c < n) tile[tx][k] = A[r + (int64_t)c * lda];
        }
        __syncthreads();
    }
    for (int k = ty; k < TB; k += 8) {
        const int r = bi * TB + tx, c = bj * TB + k;
        if (r >= n || c >= n) continue;
        E *p = A + r + (int64_t)c * lda;
        if (r == c) {
            if (mode == BX_FILL_HERM) *p = real_of(*p);
            else if (mode == BX_FILL_UNIT) *p = one_of<E>();
            continue;
        }
        if (lower ? r > c : r < c) continue; // stored element
        if (!mirror) {
            *p = zero_of<E>();
        } else {
            // A(r, c) = A(c, r) = tile[c - bj*32][r - bi*32]
            const E v = tile[k][tx];
            *p = mode == BX_FILL_HERM ? conj_of(v) : v;
        }
    }
}

// out(c, r) = op(in(r, c)) for an r x c block: 32 x 32 tiles through LDS so
// both sides coalesce; conj for the conjugate transpose
template <typename E>
__global__ __launch_bounds__(256) void k_transpose(int rows, int cols, const E *__restrict__ in,
                                                   int64_t ldi, E *__restrict__ out, int64_t ldo,
                                                   int conj)
{
    __shared__ E tile[TB][TB + 1];
    const int r0 = blockIdx.y * TB, c0 = blockIdx.x * TB;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int k = ty; k < TB; k += 8) {
        const int r = r0 + tx, c = c0 + k;
        if (r < rows && c < cols) tile[tx][k] = in[r + (int64_t)c * ldi];
    }
    __syncthreads();
    for (int k = ty; k < TB; k += 8) {
        const int c = c0 + tx, r = r0 + k; // out row c, out column r
        if (r < rows && c < cols) {
            const E v = tile[k][tx];
            out[c + (int64_t)r * ldo] = conj ? conj_of(v) : v;
        }
    }
}

// v from lane Q of each group of four lanes, to all four (DPP quad_perm
// [Q,Q,Q,Q], one move per 32-bit word)
template <int Q> __device__ __forceinline__ int quad_bcast_word(int w)
{
    return __builtin_amdgcn_update_dpp(0, w, Q * 0x55, 0xF, 0xF, false);
}
template <int Q> __device__ __forceinline__ float quad_bcast_real(float v)
{
    return __builtin_bit_cast(float, quad_bcast_word<Q>(__builtin_bit_cast(int, v)));
}
template <int Q> __device__ __forceinline__ double quad_bcast_real(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)quad_bcast_word<Q>((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)quad_bcast_word<Q>((int)(uint32_t)(u >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <int Q, typename E> __device__ __forceinline__ E quad_bcast(E v)
{
    if constexpr (is_cx<E>::value) return E{quad_bcast_real<Q>(v.re), quad_bcast_real<Q>(v.im)};
    else return quad_bcast_real<Q>(v);
}
// f(step<0>{}), ..., f(step<N-1>{}): the loop index as a compile-time
// constant, so register arrays indexed by it stay in registers
template <int V> struct step {
    static constexpr int value = V;
};
template <int K, int N, typename F> __device__ __forceinline__ void static_for(F &f)
{
    if constexpr (K < N) {
        f(step<K>{});
        static_for<K + 1, N>(f);
    }
}

// Triangular solve of one diagonal block: T (m x m, m <= NB, lower or upper,
// its own diagonal) times X = B, in place on the m x n block X.  A block of
// LEAF_THREADS threads owns LEAF_COLS columns; T and the NB x LEAF_COLS block
// of X are staged in LDS, each thread issuing all of its global loads before
// the first is waited on.  Four lanes share a column, lane q holding rows
// 4s + q (s < NB/4) in registers.  The solve runs in the loop order of
// netlib's DTRSM (Left, NoTrans: lower k = 0..m-1, upper k = m-1..0;
// x[k] /= T(k,k), then x[i] -= T(i,k) x[k] for the rows below / above): at
// step k the lane owning row k hands x[k] to its three neighbours by a quad
// broadcast, all four divide it alike, and each updates its own rows, so one
// lane does a quarter of the column's FMAs.  An upper T is staged with rows
// and columns reversed and solved as a lower one.  T is kept by step (tq[k]
// holds column k, lane q's rows contiguous) for wide LDS reads.  Rows
// m..NB-1 are padded as identity rows and never stored.
// What bounds it is the chain of NB steps, in a handful of blocks, and each
// step's reads of T.  Lane q's rows of a column lie at q (S + 1): at q S the
// four lanes' words shared banks (64 x 1024, FP64: 23.3 against 12.7 us).
// Four steps use up one register slot, and the slots move down by one; NB/16
// stretches hold 16, 12, .. slots.  (Unrolled 12.0 us, as a loop of four
// steps 12.7.)  Column k+1 of T is read during step k.  Real T(k,k) are inverted once
// per block, off the chain: x / T(k,k) is then a product and one correction
// (Markstein 1990: with r = RN(1/t) and q0 = RN(x r), RN(q0 + RN(x - q0 t) r)
// is RN(x/t)), which holds while nothing overflows or underflows.  A block in
// which a diagonal or a quotient (other than zero) leaves the safe range of
// exponents solves again with divisions.
// 64 x 1024 block, FP64: 16.2 -> 12.1 us (0.15 of them the zeros' signs).
constexpr int LEAF_THREADS = 256;
constexpr int LEAF_COLS = LEAF_THREADS / 4;

// whether v's exponent is in [-400, 400] (double), [-40, 40] (float)
__device__ __forceinline__ bool in_range(double v)
{
    const uint32_t e = ((uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32) & 0x7FFFFFFFu) >> 20;
    return e - (1023 - 400) <= 800u;
}
__device__ __forceinline__ bool in_range(float v)
{
    const uint32_t e = (__builtin_bit_cast(uint32_t, v) & 0x7FFFFFFFu) >> 23;
    return e - (127 - 40) <= 80u;
}

// a / t, r = RN(1/t); bad where it may differ from the division.  The
// remainder of a zero a is +0 whatever a's sign, so the correction would turn
// -0 / t into +0 for t > 0: the result's sign is q's.
template <typename E> __device__ __forceinline__ E quotient(E a, E t, E r, bool &bad)
{
    if constexpr (is_cx<E>::value) return divide(a, t);
    else {
        const E q = a * r;
        bad |= q == E(0) && a != E(0);
        return copysign(fma(fma(-q, t, a), r, q), q);
    }
}
template <typename E> __device__ __forceinline__ bool unsafe(E v)
{
    if constexpr (is_cx<E>::value) return false;
    else return v != E(0) && !in_range(v);
}

template <typename E, int NB>
__global__ __launch_bounds__(LEAF_THREADS) void k_trsm_leaf(int lower, int m, int n,
                                                            const E *__restrict__ T, int64_t ldt,
                                                            E *__restrict__ X, int64_t ldx)
{
    constexpr int S = NB / 4;                      // rows per lane
    constexpr int G = LEAF_THREADS / NB;           // staging: column groups
    constexpr int PT = NB / G, PX = LEAF_COLS / G; // staged columns per thread
    constexpr int Q = S + 1, P = 4 * Q;            // pitches of lanes and columns in tq
    static_assert(S * 4 == NB && S % 4 == 0 && G * NB == LEAF_THREADS && PT * G == NB &&
                      PX * G == LEAF_COLS, "leaf tiling");
    // tq[k][q*Q + s] = T(4s + q, k); reads ahead of the last column and past
    // the last slot, whose values go nowhere, stay inside the extra rows
    __shared__ E tq[NB + 2][P];
    __shared__ E xs[NB][LEAF_COLS + 1]; // xs[i][c] = X(i, j0 + c)
    __shared__ E rd[NB + 1];            // 1 / T(k, k)
    __shared__ int outside;             // a diagonal or quotient outside the safe range
    const int tid = threadIdx.x, j0 = blockIdx.x * LEAF_COLS;
    const int r = tid % NB, g = tid / NB;
    const int rs = lower ? r : NB - 1 - r; // row r's place in LDS
    auto load_x = [&](E *xv) {
#pragma unroll
        for (int p = 0; p < PX; ++p) {
            const int j = j0 + g + p * G;
            xv[p] = (r < m && j < n) ? X[r + (int64_t)j * ldx] : zero_of<E>();
        }
    };
    auto stage_x = [&](const E *xv) {
#pragma unroll
        for (int p = 0; p < PX; ++p) xs[rs][g + p * G] = xv[p];
    };
    {
        E tv[PT], xv[PX];
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const int c = g + p * G;
            tv[p] = (r < m && c < m) ? T[r + (int64_t)c * ldt]
                                     : (r == c ? one_of<E>() : zero_of<E>());
        }
        load_x(xv);
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const int c = g + p * G;
            tq[lower ? c : NB - 1 - c][(rs & 3) * Q + (rs >> 2)] = tv[p];
        }
        stage_x(xv);
    }
    if (tid == 0) outside = 0;
    __syncthreads();
    if constexpr (!is_cx<E>::value) {
        if (tid < NB) {
            const E t = tq[tid][(tid & 3) * Q + (tid >> 2)];
            rd[tid] = E(1) / t;
            if (unsafe(t) || t == E(0)) outside = 1;
        }
        __syncthreads();
    }
    const int col = tid >> 2, q = tid & 3;
    // one column solved in place in xs; whether a quotient left the safe range
    auto solve = [&](auto div_c) {
        constexpr bool DIV = is_cx<E>::value || decltype(div_c)::value;
        E x[S], tc[2][S], td[2], tr[2];
        bool bad = false;
#pragma unroll
        for (int s = 0; s < S; ++s) x[s] = xs[4 * s + q][col];
        const E *tp = &tq[0][q * Q], *dp = &tq[0][0], *rp = rd; // this slot's column, diagonal
        E *xp = &xs[q][col];
#pragma unroll
        for (int s = 0; s < S; ++s) tc[0][s] = tp[s];
        td[0] = dp[0];
        if constexpr (!DIV) tr[0] = rp[0];
        auto slots = [&](auto gc) {
            constexpr int R = S - 4 * decltype(gc)::value; // slots held
#pragma unroll
            for (int it = 0; it < 4; ++it) {
                auto one = [&](auto jc) {
                    constexpr int j = decltype(jc)::value, at = j & 1, nx = at ^ 1;
                    // column k+1, from this slot's rows on, or the next slot's
#pragma unroll
                    for (int s = 0; s < R; ++s) tc[nx][s] = tp[(j + 1) * P + (j == 3) + s];
                    td[nx] = j < 3 ? dp[(j + 1) * (P + Q)] : dp[4 * P + 1];
                    if constexpr (!DIV) tr[nx] = rp[j + 1];
                    const E xb = quad_bcast<j>(x[0]), t = td[at];
                    const E xk = DIV ? divide(xb, t) : quotient(xb, t, tr[at], bad);
                    // slot 0: row k itself on lane j, rows after it on the lanes past j
                    const E upd = sub_mul(x[0], tc[at][0], xk);
                    x[0] = pick(q == j, xk, pick(q > j, upd, x[0]));
#pragma unroll
                    for (int s = 1; s < R; ++s) x[s] = sub_mul(x[s], tc[at][s], xk);
                };
                static_for<0, 4>(one);
                *xp = x[0];
                if constexpr (!DIV) bad |= unsafe(x[0]);
#pragma unroll
                for (int s = 0; s + 1 < R; ++s) x[s] = x[s + 1];
                x[R - 1] = zero_of<E>();
                tp += 4 * P + 1, dp += 4 * P + 1, rp += 4, xp += 4 * (LEAF_COLS + 1);
            }
        };
        static_for<0, S / 4>(slots);
        return bad;
    };
    if constexpr (is_cx<E>::value) {
        solve(step<1>{});
    } else {
        const bool diag_out = outside;
        __syncthreads();
        if (!diag_out && solve(step<0>{})) outside = 1;
        __syncthreads();
        if (outside) {
            E xv[PX]; // X itself is unchanged so far
            load_x(xv);
            stage_x(xv);
            __syncthreads();
            solve(step<1>{});
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        const int c = g + p * G, j = j0 + c;
        if (r < m && j < n) X[r + (int64_t)j * ldx] = xs[rs][c];
    }
}

// dst = src on the triangle tri names (BX_TRI_* bits; row >= col for lower,
// row <= col for upper), the other triangle of dst untouched; BX_TRI_HERM
// also zeroes the diagonal's imaginary part
template <typename E>
__global__ void k_tri_copy(int n, int tri, const E *__restrict__ src, int64_t lds,
                           E *__restrict__ dst, int64_t ldd)
{
    const int64_t total = (int64_t)n * n;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(t % n), c = (int)(t / n);
        if ((tri & BX_TRI_LOWER) ? r < c : r > c) continue;
        E v = src[r + (int64_t)c * lds];
        if ((tri & BX_TRI_HERM) && r == c) v = real_of(v);
        dst[r + (int64_t)c * ldd] = v;
    }
}

template <typename E, int NB>
void launch_leaf(dim3 grid, int lower, int m, int n, const void *T, int64_t ldt, void *X, int64_t ldx,
                 hipStream_t st)
{
    hipLaunchKernelGGL((k_trsm_leaf<E, NB>), grid, dim3(LEAF_THREADS), 0, st, lower, m, n,
                       (const E *)T, ldt, (E *)X, ldx);
}

template <typename E> int launch_fill(int n, int lower, int mode, void *A, int64_t lda, hipStream_t st)
{
    const int nt = (n + TB - 1) / TB;
    hipLaunchKernelGGL(k_tri_fill<E>, dim3(nt, nt), dim3(256), 0, st, n, lower, mode, (E *)A, lda);
    return hipGetLastError() == hipSuccess ? 0 : BLASX_EHIP;
}

} // namespace

extern "C" {

int bxh_tri_fill(int dtype, int n, int lower, int mode, void *A, int64_t lda, void *stream)
{
    if (n <= 0) return 0;
    if (lda < n || mode < BX_FILL_SYM || mode > BX_FILL_UNIT) return BLASX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
    case BLASX_S: return launch_fill<float>(n, lower, mode, A, lda, st);
    case BLASX_D: return launch_fill<double>(n, lower, mode, A, lda, st);
    case BLASX_Z: return launch_fill<z16>(n, lower, mode, A, lda, st);
    case BLASX_C: return launch_fill<c8>(n, lower, mode, A, lda, st);
    default: return BLASX_EINVAL;
    }
}

int bxh_transpose(int dtype, int rows, int cols, const void *in, int64_t ldi, void *out, int64_t ldo,
                  int conj, void *stream)
{
    if (rows <= 0 || cols <= 0) return 0;
    const dim3 grid((cols + TB - 1) / TB, (rows + TB - 1) / TB);
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
    case BLASX_S:
        hipLaunchKernelGGL(k_transpose<float>, grid, dim3(256), 0, st, rows, cols,
                           (const float *)in, ldi, (float *)out, ldo, 0);
        break;
    case BLASX_D:
        hipLaunchKernelGGL(k_transpose<double>, grid, dim3(256), 0, st, rows, cols,
                           (const double *)in, ldi, (double *)out, ldo, 0);
        break;
    case BLASX_Z:
        hipLaunchKernelGGL(k_transpose<z16>, grid, dim3(256), 0, st, rows, cols, (const z16 *)in,
                           ldi, (z16 *)out, ldo, conj);
        break;
    case BLASX_C:
        hipLaunchKernelGGL(k_transpose<c8>, grid, dim3(256), 0, st, rows, cols, (const c8 *)in,
                           ldi, (c8 *)out, ldo, conj);
        break;
    default: return BLASX_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? 0 : BLASX_EHIP;
}

int bxh_trsm_leaf_nb(int dtype) { return dtype == BLASX_Z ? 32 : 64; }


int bxh_trsm_leaf(int dtype, int lower, int m, int n, const void *T, int64_t ldt, void *X,
                  int64_t ldx, void *stream)
{
    const int nb = bxh_trsm_leaf_nb(dtype);
    if (m <= 0 || n <= 0) return 0;
    if (m > nb || ldt < m || ldx < m) return BLASX_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((n + LEAF_COLS - 1) / LEAF_COLS);
    switch (dtype) {
    case BLASX_S: launch_leaf<float, 64>(grid, lower, m, n, T, ldt, X, ldx, st); break;
    case BLASX_D: launch_leaf<double, 64>(grid, lower, m, n, T, ldt, X, ldx, st); break;
    case BLASX_Z: launch_leaf<z16, 32>(grid, lower, m, n, T, ldt, X, ldx, st); break;
    case BLASX_C: launch_leaf<c8, 64>(grid, lower, m, n, T, ldt, X, ldx, st); break;
    default: return BLASX_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? 0 : BLASX_EHIP;
}

int bxh_tri_copy(int dtype, int n, int tri, const void *src, int64_t lds, void *dst, int64_t ldd,
                 void *stream)
{
    if (n <= 0) return 0;
    const int64_t total = (int64_t)n * n;
    int grid = (int)((total + 255) / 256);
    if (grid > 65536) grid = 65536;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
    case BLASX_S:
        hipLaunchKernelGGL(k_tri_copy<float>, dim3(grid), dim3(256), 0, st, n, tri,
                           (const float *)src, lds, (float *)dst, ldd);
        break;
    case BLASX_D:
        hipLaunchKernelGGL(k_tri_copy<double>, dim3(grid), dim3(256), 0, st, n, tri,
                           (const double *)src, lds, (double *)dst, ldd);
        break;
    case BLASX_Z:
        hipLaunchKernelGGL(k_tri_copy<z16>, dim3(grid), dim3(256), 0, st, n, tri,
                           (const z16 *)src, lds, (z16 *)dst, ldd);
        break;
    case BLASX_C:
        hipLaunchKernelGGL(k_tri_copy<c8>, dim3(grid), dim3(256), 0, st, n, tri, (const c8 *)src,
                           lds, (c8 *)dst, ldd);
        break;
    default: return BLASX_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? 0 : BLASX_EHIP;
}

int bxh_memcpy2d_d2d_async(void *dst, size_t dpitch, const void *src, size_t spitch, size_t width,
                           size_t height, void *s)
{
    if (!width || !height) return 0;
    const hipError_t e = hipMemcpy2DAsync(dst, dpitch, src, spitch, width, height,
                                          hipMemcpyDeviceToDevice, (hipStream_t)s);
    return e == hipSuccess ? 0 : BLASX_EHIP;
}

} // extern "C"
