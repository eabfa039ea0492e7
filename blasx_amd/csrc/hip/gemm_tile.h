// gemm_tile.h -- the GEMM block tiles (gfx950): C = alpha sum_s op(A_s)
// op(B_s) + beta C for FP32, FP64 and complex128 (four FP64 products per
// complex one, the signs of conjugation and of the real part by the MFMA's
// NEG modifier).  The reference hands the same product to cuBLAS
// (blas/blasx_dgemm.c:87-94, blas/blasx_sgemm.c:87, blas/blasx_zgemm.c:88).
//
// 256 threads, 2x2 waves of WTM x WTN, five block shapes: 32x32, 64x32, 64x64,
// 128x64 and 128x128 (FP64, and FP32 in grouped launches).  What bounds a tile is the matrix core's issue: one FP64 MFMA
// takes 64 cycles of its SIMD (FP32: 32), back to back even in one dependent
// chain, and every vector ALU instruction beside it takes its slot.  So the K
// loop has none: operand addresses are scalar bases plus constant lane
// offsets, the LDS stage of each step is an immediate (the loop is unrolled
// over the stages), the DMA moves global memory to LDS without registers, and
// the fragment reads of half a K tile are spread over the products of the
// other half.  Measured at 4096^3, FP64, 64x64 tiles: 66 TFLOP/s with
// per-step address arithmetic, 74.5 without (the MFMA alone: 78); one block
// on a CU alone takes 458 ns per K tile of 16, 432 of them MFMAs.
// The same order of K in every shape and movement: all give the same bits.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"

namespace {

// 16-byte chunks: EPC elements each; a K tile is KT values of K, 8 chunks
// (128 bytes) per row in either layout.
template <typename E> struct Chunk {
    static constexpr int EPC = 16 / (int)sizeof(E), KT = 128 / (int)sizeof(E);
};

// the K value lane group lg (lane / 16) feeds at K step s of a K tile: the
// same order in every kernel, so that all sum a C element's products alike
template <typename E> __device__ __forceinline__ constexpr int step_k(int s, int lg)
{
    if constexpr (sizeof(E) == 16) return 4 * s + lg;
    else if constexpr (sizeof(E) == 8) return 2 * (4 * (s >> 1) + lg) + (s & 1);
    else return 4 * (lg + 4 * (s >> 2)) + (s & 3);
}

// One operand's stage: ROWS x KT elements as 16-byte chunks.
//  MAJ_MN (rows contiguous in memory): chunk (k, row / EPC) at position
//  (k ROWS / EPC + row / EPC) ^ swz(k), swz chosen so that the lane groups
//  of one fragment read, whose k differ, fall on different banks;
//  MAJ_K: chunk (row, k / EPC) at position 8 row + ((k / EPC) ^ ((row >> 1) & 7)).
// The XOR touches only bits that the mask does not depend on, so it is its
// own inverse.
template <typename E, int MAJ, int ROWS> struct Stage {
    static constexpr int EPC = Chunk<E>::EPC, KT = Chunk<E>::KT;
    static constexpr int CPK = ROWS / EPC;    // chunks per k (MAJ_MN)
    static constexpr int ELEMS = ROWS * KT;
    static constexpr int NI = ROWS * 8 / NT;  // chunks per thread

    static __device__ __forceinline__ int swz(int k)
    {
        if constexpr (sizeof(E) == 8) return ((k >> 1) & 1) << 3;
        else if constexpr (sizeof(E) == 4) return ((k >> 2) & 3) << 2;
        else return 0;
    }
    // the operand element at the start of chunk p of the stage
    static __device__ __forceinline__ void source(int p, int &row, int &k)
    {
        if constexpr (MAJ == MAJ_MN) {
            const int idx = p ^ swz(p / CPK);
            k = idx / CPK;
            row = (idx % CPK) * EPC;
        } else {
            row = p >> 3;
            k = ((p & 7) ^ ((row >> 1) & 7)) * EPC;
        }
    }
    // position of element (row, k), in elements
    static __device__ __forceinline__ int at(int row, int k)
    {
        if constexpr (MAJ == MAJ_MN)
            return ((k * CPK + row / EPC) ^ swz(k)) * EPC + row % EPC;
        else
            return (row * 8 + ((k / EPC) ^ ((row >> 1) & 7))) * EPC + k % EPC;
    }
};

// 16 bytes per lane from global memory to LDS at lds + 16 lane (`lds`
// wave-uniform).  M0 is reserved: the compiler does not allocate it, and
// nothing else in these kernels uses it.  A load to LDS may read the old M0 in
// the cycle after a scalar write of it: one wait state between them, which the
// compiler does not put inside inline assembly.
__device__ __forceinline__ void dma16_lds(const void *base, uint32_t off, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(off), "s"(base)
                 : "memory");
}
// S_WAITCNT with the LDS counter at 0, and with the vector-memory counter at N;
// by the builtin, so that the compiler's own waits know what has arrived
__device__ __forceinline__ void lds_wait() { __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4)); }
template <int N> __device__ __forceinline__ void vm_wait()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
// all but N vector-memory operations and every LDS operation of this wave are
// done; then all waves of the block meet.  No access moves across.
// (N < 0: no wait for vector-memory operations)
template <int N> __device__ __forceinline__ void wait_meet()
{
    asm volatile("" : : : "memory");
    lds_wait();
    if constexpr (N >= 0) vm_wait<N>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
}

typedef uint32_t u32x4_e __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_l __attribute__((ext_vector_type(4)));

// One operand of a block tile: DMA = true moves 16-byte aligned chunks from
// global memory straight to LDS; DMA = false loads 16 bytes at element
// alignment into registers and stores them to the same LDS positions.  Each
// of a wave's NI loads has a scalar base, advanced by scalar adds, and a
// 32-bit lane offset, which covers at most 8 rows or K values: the host
// checks 8 ld sizeof(E) < 2^32.
template <typename E, int MAJ, int ROWS, bool DMA> struct Mover {
    typedef Stage<E, MAJ, ROWS> S_;
    static constexpr int NI = S_::NI, EPC = S_::EPC, BK = Chunk<E>::KT;
    static constexpr int TAIL = ROWS * BK / NT;
    // LDS reads of a wave's fragments for half a K tile, ROWS / 32 blocks of 16 rows
    static constexpr int READS = ROWS / 32 * (BK / 8) / (MAJ == MAJ_K ? EPC : 1);
    const char *base[NI];
    uint32_t off[NI];
    int64_t step; // bytes from one K tile to the next
    u32x4_l reg[DMA ? 1 : NI];
    int shift[(!DMA && MAJ == MAJ_MN) ? NI : 1];
    bool edge;
    E tail[TAIL];

    // rows r0 .. of an operand of rlim rows.  Rows past the last are read
    // from the last one(s): they feed only outputs that are not written.
    __device__ __forceinline__ void init(const E *X, int64_t ld, int r0, int rlim, int tid)
    {
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        step = (MAJ == MAJ_MN ? (int64_t)BK * ld : (int64_t)BK) * (int64_t)sizeof(E);
        edge = !DMA && MAJ == MAJ_MN && r0 + ROWS > rlim;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            // a wave's load fills 64 consecutive chunks
            int row, k;
            S_::source(i * NT + tid, row, k);
            const int g = r0 + row;
            if constexpr (MAJ == MAJ_K) {
                const int b = min(r0 + (i * NT + wave * 64) / 8, rlim - 1);
                base[i] = (const char *)(X + (int64_t)b * ld);
                off[i] = ((uint32_t)(min(g, rlim - 1) - b) * (uint32_t)ld + k) * (uint32_t)sizeof(E);
            } else {
                // DMA: stays in the 16-byte granule of the last row (aligned
                // ld); else inside the column, the last EPC rows (rlim >= EPC)
                const int last = DMA ? (rlim - 1) & ~(EPC - 1) : rlim - EPC;
                const int c = min(g, last), b = min(r0, last), kb = (i * NT + wave * 64) / S_::CPK;
                if constexpr (!DMA) shift[i] = min(g - c, EPC - 1);
                base[i] = (const char *)(X + b + (int64_t)kb * ld);
                off[i] = ((uint32_t)(k - kb) * (uint32_t)ld + (c - b)) * (uint32_t)sizeof(E);
            }
        }
    }
    __device__ __forceinline__ void dma(uint32_t lds)
    {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            dma16_lds(base[i], off[i], lds + i * NT * 16);
            base[i] += step;
        }
    }
    __device__ __forceinline__ void load()
    {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            // opaque here, so that the 32-bit offset goes into the load
            // itself instead of 64-bit vector adds on every step
            uint32_t o = off[i];
            asm volatile("" : "+v"(o));
            reg[i] = *(const __attribute__((address_space(1))) u32x4_e *)(
                (const __attribute__((address_space(1))) char *)base[i] + o);
            base[i] += step;
        }
    }
    __device__ __forceinline__ void store(E *stage, int tid)
    {
        if constexpr (MAJ == MAJ_MN && EPC > 1) {
            if (edge) {
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    if constexpr (EPC == 2) {
                        if (shift[i]) reg[i].xy = reg[i].zw;
                    } else {
                        if (shift[i] & 1) reg[i].xyz = reg[i].yzw;
                        if (shift[i] & 2) reg[i].xy = reg[i].zw;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
            *(u32x4_l *)(stage + (i * NT + tid) * EPC) = reg[i];
    }
    // Element i of this thread's share of kr <= BK columns of K, from k0:
    // zero beyond, so that the extra products add nothing.
    static __device__ __forceinline__ void tail_at(int i, int tid, int &row, int &k)
    {
        const int e = tid + i * NT;
        row = MAJ == MAJ_MN ? e % ROWS : e / BK;
        k = MAJ == MAJ_MN ? e / ROWS : e % BK;
    }
    static __device__ __forceinline__ E tail_load(const E *X, int64_t ld, int r0, int rlim,
                                                  int64_t k0, int kr, int row, int k)
    {
        if (k >= kr || r0 + row >= rlim) return zero_of<E>();
        return gload(X + (MAJ == MAJ_MN ? (r0 + row) + (k0 + k) * ld
                                        : (k0 + k) + (int64_t)(r0 + row) * ld));
    }
    __device__ __forceinline__ void load_tail(const E *X, int64_t ld, int r0, int rlim, int64_t k0,
                                              int kr, int tid)
    {
#pragma unroll
        for (int i = 0; i < TAIL; ++i) {
            int row, k;
            tail_at(i, tid, row, k);
            tail[i] = tail_load(X, ld, r0, rlim, k0, kr, row, k);
        }
    }
    __device__ __forceinline__ void store_tail(E *stage, int tid)
    {
#pragma unroll
        for (int i = 0; i < TAIL; ++i) {
            int row, k;
            tail_at(i, tid, row, k);
            stage[S_::at(row, k)] = tail[i];
        }
    }
    // both, four elements at a time (fewer registers)
    static __device__ __forceinline__ void copy_tail(const E *X, int64_t ld, int r0, int rlim,
                                                     int64_t k0, int kr, E *stage, int tid)
    {
        constexpr int STEP = TAIL < 4 ? TAIL : 4;
#pragma unroll 1
        for (int i0 = 0; i0 < TAIL; i0 += STEP) {
            E v[STEP];
#pragma unroll
            for (int i = 0; i < STEP; ++i) {
                int row, k;
                tail_at(i0 + i, tid, row, k);
                v[i] = tail_load(X, ld, r0, rlim, k0, kr, row, k);
            }
#pragma unroll
            for (int i = 0; i < STEP; ++i) {
                int row, k;
                tail_at(i0 + i, tid, row, k);
                stage[S_::at(row, k)] = v[i];
            }
        }
    }
};

// the fragments of NB 16-row blocks (rows row0 + 16 i) for the GS K steps
// from q0 of a stage, whole 16-byte chunks at a time where a chunk runs along K
template <typename S_, int MAJ, int GS, int NB, typename E>
__device__ __forceinline__ void read_frags(E (&f)[GS][NB], const E *st, int row0, int lg, int q0)
{
    constexpr int PER = MAJ == MAJ_K ? S_::EPC : 1;
#pragma unroll
    for (int q = 0; q < GS; q += PER)
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const E *p = st + S_::at(row0 + i * 16, step_k<E>(q0 + q, lg));
            if constexpr (PER == 1) {
                f[q][i] = *p;
            } else {
                struct alignas(16) V {
                    E e[PER];
                } v = *(const V *)p;
#pragma unroll
                for (int e = 0; e < PER; ++e) f[q + e][i] = v.e[e];
            }
        }
}

template <int V> struct Int {
    static constexpr int value = V;
};

// v_mfma_f64 with the negations its NEG modifier gives for free: bit 0 the
// first operand, bit 1 the second
template <int NEG> __device__ __forceinline__ d4_t mfma_neg(double a, double b, d4_t c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, NEG);
}

// Block tile of 2x2 waves, each WTM x WTN, with NS LDS stages.
template <typename E, int WTM, int WTN, int NS> struct Shape {
    static constexpr int BM = 2 * WTM, BN = 2 * WTN;
    static constexpr int SMEM = NS * (BM + BN) * 128;
};

template <typename E, int MAJA, int MAJB, bool CJA, bool CJB, int WTM, int WTN, int NS, bool DMA>
__device__ __forceinline__ void tile_block(const bxh_problem_t &P, const bxh_seg_t *segs,
                                           const bxh_seg_t &seg0, const bxh_seg_t &seg1, int tm,
                                           int tn, char *smem)
{
    typedef Shape<E, WTM, WTN, NS> H;
    typedef Mover<E, MAJA, H::BM, DMA> MA;
    typedef Mover<E, MAJB, H::BN, DMA> MB;
    constexpr bool CPLX = sizeof(E) == 16;
    constexpr int FM = WTM / 16, FN = WTN / 16, BK = Chunk<E>::KT;
    constexpr int GS = BK / 8, ALL = GS * FM; // K steps and products (times FN) per half tile
    typedef typename Cfg<E>::acc_t acc_t;
    // opaque: a kernel that holds several blocks would otherwise compute all
    // their lane addresses before choosing one
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    tid &= NT - 1;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1, l16 = lane & 15, lg = lane >> 4;
    const int m0 = tm * H::BM, n0 = tn * H::BN;
    E *sA = (E *)smem, *sB = sA + NS * MA::S_::ELEMS;
    auto stA = [&](int s) { return sA + s * MA::S_::ELEMS; };
    auto stB = [&](int s) { return sB + s * MB::S_::ELEMS; };
    const uint32_t lA = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)sA + wave * 1024);
    const uint32_t lB = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)sB + wave * 1024);

    // acc[i][j]: rows 16 i + l16 of the wave's part of C, columns 16 j +
    // out_row(lg, v): the B fragment is the MFMA's row operand, so that 16
    // lanes hold 16 consecutive rows of a column of C
    acc_t acc[FM][FN][CPLX ? 2 : 1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int c = 0; c < (CPLX ? 2 : 1); ++c) acc[i][j][c] = acc_t{0, 0, 0, 0};

    // the fragments of half a staged K tile (h = 0, 1), and its products [x0,
    // x1) of GS FM (K step, row block) pairs
    struct Frags {
        E a[GS][FM], b[GS][FN];
    };
    auto read = [&](Frags &f, int s, int h) {
        read_frags<typename MA::S_, MAJA, GS, FM>(f.a, stA(s), wm * WTM + l16, lg, h * GS);
        read_frags<typename MB::S_, MAJB, GS, FN>(f.b, stB(s), wn * WTN + l16, lg, h * GS);
    };
    auto products = [&](const Frags &f, int x0, int x1) {
#pragma unroll
        for (int x = 0; x < ALL; ++x) {
            if (x < x0 || x >= x1) continue;
            const int q = x / FM, i = x % FM;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (CPLX) {
                    const cplx a = f.a[q][i], b = f.b[q][j];
                    acc[i][j][0] = mfma(b.re, a.re, acc[i][j][0]);
                    acc[i][j][1] = mfma_neg<CJB ? 1 : 0>(b.im, a.re, acc[i][j][1]);
                    acc[i][j][0] = mfma_neg<CJA == CJB ? 2 : 0>(b.im, a.im, acc[i][j][0]);
                    acc[i][j][1] = mfma_neg<CJA ? 2 : 0>(b.re, a.im, acc[i][j][1]);
                } else {
                    acc[i][j][0] = mfma(f.b[q][j], f.a[q][i], acc[i][j][0]);
                }
            }
        }
    };
    // spreads the LDS reads of a half over mf products: in one run they
    // would leave the matrix core idle
    auto spread = [&](auto mf_c) {
        constexpr int MF = decltype(mf_c)::value, RD = MA::READS + MB::READS;
        constexpr int PER = MF ? (RD + MF - 1) / MF : 1;
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, PER, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    for (int si = 0; si < P.nseg; ++si) {
        const bxh_seg_t sg = seg_at(segs, seg0, seg1, si);
        if (sg.k <= 0) continue;
        const E *A = (const E *)sg.A, *B = (const E *)sg.B;
        const int T = !DMA && P.form == BXH_FORM_ELEMENT ? 0 : (int)(sg.k / BK);
        const int kr = (int)min((int64_t)BK, sg.k - (int64_t)T * BK);
        MA ma;
        MB mb;
        // the last K columns: loaded before the K loop where registers allow
        constexpr bool EARLY = DMA && FM * FN <= 4;
        if (EARLY && kr) {
            ma.load_tail(A, sg.lda, m0, P.m, (int64_t)T * BK, kr, tid);
            mb.load_tail(B, sg.ldb, n0, P.n, (int64_t)T * BK, kr, tid);
        }
        ma.init(A, sg.lda, m0, P.m, tid);
        mb.init(B, sg.ldb, n0, P.n, tid);
        constexpr int IPT = MA::NI + MB::NI;
        constexpr uint32_t STA = MA::S_::ELEMS * sizeof(E), STB = MB::S_::ELEMS * sizeof(E);
        // Tile t in stage t % NS.  When step t begins, the first half of its
        // fragments is in registers; the second half is read under the first
        // half's products.  After the first FIRST of the second half's
        // products the wave has read the whole tile, and meets the other
        // waves: stage t % NS is then free.
        //  DMA: tile t + NS goes there; the wave first waits for its part of
        //  tile t + 1 (the NS - 2 tiles after it may be in flight).
        //  else (NS = 2): tile t + 2, loaded into registers a step ago, is
        //  stored there and tile t + 3's loads start.
        // Tile t + 1's first half is read under the other products.
        constexpr int FIRST = GS > 1 ? FM : FM / 2, MPX = FN * (CPLX ? 4 : 1);
        static_assert(DMA || NS == 2, "register-staged: two LDS stages");
        if constexpr (DMA) {
#pragma unroll
            for (int t = 0; t < NS; ++t)
                if (t < T) {
                    ma.dma(lA + t * STA);
                    mb.dma(lB + t * STB);
                }
            if (T >= NS) wait_meet<IPT * (NS - 1)>();
            else wait_meet<0>();
        } else {
#pragma unroll
            for (int t = 0; t < 3; ++t)
                if (t < T) {
                    ma.load();
                    mb.load();
                    if (t < 2) {
                        ma.store(stA(t), tid);
                        mb.store(stB(t), tid);
                    }
                }
            wait_meet<-1>();
        }
        Frags f0, f1;
        int t = 0;
        if (T > 0) read(f0, 0, 0);
        // one step with its stage as a constant: the LDS addresses are then
        // immediates, and the step has no vector ALU instruction, each of
        // which would take the matrix core's issue slot
        auto step = [&](auto u_c, auto full_c) {
            constexpr int s = decltype(u_c)::value, n = (s + 1) % NS;
            constexpr bool FULL = decltype(full_c)::value;
            read(f1, s, 1);
            products(f0, 0, ALL);
            spread(Int<ALL * MPX>{});
            products(f1, 0, FIRST);
            __builtin_amdgcn_sched_barrier(0);
            lds_wait(); // on every path: no later wait is for these reads
            if (FULL || t + 1 < T) {
                if constexpr (DMA) {
                    if (FULL || t + NS < T) {
                        wait_meet<IPT *(NS - 2)>();
                        ma.dma(lA + s * STA);
                        mb.dma(lB + s * STB);
                    } else {
                        wait_meet<0>();
                    }
                } else {
                    wait_meet<-1>();
                    if (FULL || t + 2 < T) {
                        ma.store(stA(s), tid);
                        mb.store(stB(s), tid);
                    }
                    if (FULL || t + 3 < T) {
                        ma.load();
                        mb.load();
                    }
                }
                read(f0, n, 0);
            }
            products(f1, FIRST, ALL);
            if constexpr (FULL) spread(Int<(ALL - FIRST) * MPX>{});
            ++t;
        };
        constexpr int U = NS, AHEAD = DMA ? NS : 3;
        static_assert(U >= 2 && U <= 4, "steps per unrolled loop");
        auto steps = [&](auto full_c) {
            constexpr bool FULL = decltype(full_c)::value;
            step(Int<0>{}, full_c);
            if (FULL || t < T) step(Int<1>{}, full_c);
            if constexpr (U > 2)
                if (FULL || t < T) step(Int<2>{}, full_c);
            if constexpr (U > 3)
                if (FULL || t < T) step(Int<3>{}, full_c);
        };
        while (t + U + AHEAD <= T) steps(Int<1>{});
        while (t < T) steps(Int<0>{});
        for (int64_t k0 = (int64_t)T * BK; k0 < sg.k; k0 += BK) {
            const int kt = (int)min((int64_t)BK, sg.k - k0);
            __syncthreads(); // stage 0 is free
            if constexpr (EARLY) {
                ma.store_tail(stA(0), tid);
                mb.store_tail(stB(0), tid);
            } else {
                MA::copy_tail(A, sg.lda, m0, P.m, k0, kt, stA(0), tid);
                MB::copy_tail(B, sg.ldb, n0, P.n, k0, kt, stB(0), tid);
            }
            __syncthreads();
            for (int h = 0; h < 2; ++h) {
                read(f0, 0, h);
                products(f0, 0, ALL);
            }
        }
        if (P.nseg > 1) __syncthreads(); // the next segment reuses the stages
    }

    E *Cp = (E *)P.C;
    const int tri = P.tri, toff = P.tri_off;
    const bool bz = P.beta_zero;
    const int row0 = m0 + wm * WTM + l16, col0 = n0 + wn * WTN;
    auto result = [&](int i, int j, int v, E c0) {
        if constexpr (CPLX)
            return out_cplx(P.alpha_re, P.alpha_im, acc[i][j][0][v], acc[i][j][1][v], P.beta_re,
                            P.beta_im, c0, bz);
        else
            return out_real((E)P.alpha_re, acc[i][j][0][v], (E)P.beta_re, c0, bz);
    };
    if (!tri && m0 + H::BM <= P.m && n0 + H::BN <= P.n) {
        // a whole tile: 16 loads of C are issued before the first store
        constexpr int JN = FM * FN <= 4 ? FN : 16 / (4 * FM);
        E *c = Cp + row0 + (int64_t)col0 * P.ldc;
#pragma unroll
        for (int j0 = 0; j0 < FN; j0 += JN) {
            E c0[JN][4][FM];
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
                        c0[j][v][i] = bz ? zero_of<E>()
                                         : gload(c + i * 16 + (int64_t)((j0 + j) * 16 + Cfg<E>::out_row(lg, v)) * P.ldc);
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int i = 0; i < FM; ++i)
                        gstore(c + i * 16 + (int64_t)((j0 + j) * 16 + Cfg<E>::out_row(lg, v)) * P.ldc,
                               result(i, j0 + j, v, c0[j][v][i]));
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = row0 + i * 16, col = col0 + j * 16 + Cfg<E>::out_row(lg, v);
                if (row >= P.m || col >= P.n || !tri_keep(tri, row + toff, col)) continue;
                E *c = Cp + row + (int64_t)col * P.ldc;
                E o = result(i, j, v, bz ? zero_of<E>() : gload(c));
                if constexpr (CPLX)
                    if ((tri & BX_TRI_HERM) && row + toff == col) o.im = 0.0;
                gstore(c, o);
            }
}

// blocks go to the 8 XCDs round-robin: XCD x takes a contiguous range of
// tiles, so that its blocks share operand panels in its L2
__device__ __forceinline__ int xcd_tile()
{
    const int nb = gridDim.x, x = blockIdx.x & 7, q = nb >> 3, r = nb & 7;
    return x * q + (x < r ? x : r) + (blockIdx.x >> 3);
}

} // namespace
