"""Block tile shapes and operand movements of the plain device GEMM.

Integer inputs whose every partial sum is exact in the element type, so the
result must equal the naive oracle bit for bit at each tile's edges, at every
remainder of K, and for each way the operands are moved: 16-byte aligned,
element aligned (odd leading dimension, offset base), and with fewer rows
than one 16-byte load takes.
"""
import ctypes as C
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


def _ints(rng, dt, shape, m):
    x = rng.integers(-m, m + 1, shape)
    if np.dtype(dt).kind == "c":
        x = x + 1j * rng.integers(-m, m + 1, shape)
    return np.asfortranarray(x.astype(dt))


def _run(bx, orc, dt, ta, tb, M, N, K, pad, off, seed):
    rng = np.random.default_rng(seed)
    cplx = np.dtype(dt).kind == "c"
    m = 8 if dt == np.float32 else 64
    ra, ca = (M, K) if ta == "N" else (K, M)
    rb, cb = (K, N) if tb == "N" else (N, K)
    A, B, C0 = (_ints(rng, dt, s, m) for s in ((ra + pad, ca), (rb + pad, cb), (M + pad, N)))
    al, be = (2 - 1j, 1 + 3j) if cplx else (3.0, -2.0)
    ref = C0.copy(order="F")
    orc.gemm(ta, tb, M, N, K, al, A, ra + pad, B, rb + pad, be, ref, M + pad)
    es = np.dtype(dt).itemsize
    dA, dB = (bx.DeviceArray.from_host(np.concatenate([np.zeros(off, dt), x.ravel(order="F")])[:, None])
              for x in (A, B))
    dC = bx.DeviceArray.from_host(C0)
    bx.device_gemm(ta, tb, M, N, K, al, dA.ptr + off * es, ra + pad, dB.ptr + off * es, rb + pad, be,
                   dC.ptr, M + pad, dt)
    bx.synchronize()
    out = dC.download()
    for d in (dA, dB, dC):
        d.free()
    assert np.array_equal(out, ref), (np.dtype(dt).name, ta, tb, M, N, K, pad, off)


# (M, N, K): one below, at and above the edges of the 32, 64 and 128 row tiles
# and of the K tiles (32 FP32, 16 FP64, 8 complex), K shorter than the pipeline
# and longer.  The library takes 32x32 and 64x32 tiles for these; the test of
# given shapes below runs the others.
SHAPES = [(1, 1, 1), (2, 3, 5), (31, 33, 7), (32, 32, 32), (33, 31, 65), (63, 65, 129), (64, 64, 64),
          (65, 129, 31), (96, 40, 1000), (129, 127, 48), (700, 600, 40), (1030, 515, 33),
          (1300, 1500, 24)]


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.complex128])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 0), (4, 1)])
def test_tile_edges_integer_exact(gpu, orc, dt, pad, off):
    ops = ([("N", "N"), ("C", "T"), ("T", "C"), ("N", "C"), ("C", "N")] if np.dtype(dt).kind == "c"
           else [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
    for i, (M, N, K) in enumerate(SHAPES):
        for ta, tb in ops if M * N < 200000 else ops[i % 2::2]:
            say("tile", np.dtype(dt).name, ta, tb, M, N, K, pad, off)
            _run(gpu, orc, dt, ta, tb, M, N, K, pad, off, 7 * i + pad)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_large_tile_integer_exact(gpu, orc, dt):
    """ragged in both dimensions, on the shape that the library takes for it: 128
    x 64 in FP64, 64 x 32 in FP32"""
    for ta, tb in (("N", "N"), ("T", "T")):
        M, N, K = 4100, 4036, 100
        say("large tile", np.dtype(dt).name, ta, tb, M, N, K)
        rng = np.random.default_rng(3)
        A, B = (_ints(rng, dt, s, 8) for s in ((M, K) if ta == "N" else (K, M), (K, N) if tb == "N" else (N, K)))
        opa, opb = (A if ta == "N" else A.T), (B if tb == "N" else B.T)
        dA, dB = gpu.DeviceArray.from_host(A), gpu.DeviceArray.from_host(B)
        dC = gpu.DeviceArray.from_host(np.full((M, N), np.nan, dt, order="F"))
        gpu.device_gemm(ta, tb, M, N, K, 1.0, dA.ptr, A.shape[0], dB.ptr, B.shape[0], 0.0, dC.ptr, M, dt)
        gpu.synchronize()
        # integers below 2^24 whatever the order: exact in the element type
        assert np.array_equal(dC.download(), (opa.astype(np.float64) @ opb.astype(np.float64)).astype(dt))
        for d in (dA, dB, dC):
            d.free()


def _tile_fn(bx):
    T = bx.test_lib()
    vp, i64 = C.c_void_p, C.c_int64
    T.bxtest_gemm_tile.argtypes = [C.c_int] * 8 + [vp, vp, i64, vp, i64, vp, i64, vp, vp, i64]
    return T.bxtest_gemm_tile


def _pair(v):
    return (C.c_double * 2)(complex(v).real, complex(v).imag)


DT = {"S": np.float32, "D": np.float64, "Z": np.complex128}
# (type, padding, offset) -> shapes: by DMA with both 0, else through registers
# (a complex operand is misaligned by its base alone: half an element)
KINDS = [("S", 0, 0, 4), ("S", 1, 0, 3), ("D", 0, 0, 5), ("D", 1, 0, 3), ("Z", 0, 0, 4),
         ("Z", 0, 8, 3)]
GIVEN = [(t, pad, off, s) for t, pad, off, n in KINDS for s in range(n)]
ROWS = [32, 64, 64, 128, 128]


def _operand(bx, x, off):
    """x in HBM `off` bytes past a 16-byte boundary, and its address"""
    raw = np.concatenate([np.zeros(off, np.uint8), x.ravel(order="F").view(np.uint8),
                          np.zeros(-(off + x.nbytes) % 8, np.uint8)])
    d = bx.DeviceArray.from_host(raw.view(np.float64)[:, None])
    return d, d.ptr + off


def _even(n, dt, pad):
    """n rounded up to a 16-byte multiple of elements, plus pad"""
    per = max(16 // np.dtype(dt).itemsize, 1)
    return -(-n // per) * per + pad


@pytest.mark.parametrize("t,pad,off,shape", GIVEN)
def test_given_tile_integer_exact(gpu, t, pad, off, shape):
    """each compiled shape and movement on products around its tile edges and on
    a grid of several tile groups, every transposition; NaN in the C that beta =
    0 must not read"""
    bx, dt = gpu, DT[t]
    fn, code = _tile_fn(bx), bx.dtype_code(dt)
    e, cplx = ROWS[shape], t == "Z"
    ops = [(a, b) for a in range(3 if cplx else 2) for b in range(3 if cplx else 2)]
    op = (lambda x: x, lambda x: x.T, lambda x: x.conj().T)
    rng = np.random.default_rng(shape)
    for M, N, K in [(e, e, 64), (e - 1, e + 1, 47), (2 * e + 1, e - 1, 9), (5, 3, 131),
                    (9 * e + 7, 3 * e + 5, 39), (3 * e, 21 * e, 96)]:
        al, be = (2 - 1j, 1 + 3j) if cplx else (3.0, -2.0)
        for j, (oa, ob) in enumerate(ops if M * N < 40000 else ops[shape % 2::2]):
            say("given tile", t, pad, off, shape, M, N, K, oa, ob)
            b0 = j % 2 == 1
            m = 4 if t == "S" else 64
            sa, sb = ((M, K) if oa == 0 else (K, M)), ((K, N) if ob == 0 else (N, K))
            lda, ldb = _even(sa[0], dt, pad), _even(sb[0], dt, pad)
            A, B, C0 = (_ints(rng, dt, x, m) for x in ((lda, sa[1]), (ldb, sb[1]), (M + pad, N)))
            prod = op[oa](A[:sa[0]]) @ op[ob](B[:sb[0]])  # exact in the element type
            ref = C0.copy(order="F")
            ref[:M] = al * prod + (0 if b0 else be * C0[:M])
            if b0:
                C0[:M] = np.nan
            (dA, pA), (dB, pB) = _operand(bx, A, off), _operand(bx, B, off)
            dC = bx.DeviceArray.from_host(C0)
            rc = fn(code, shape, 0, oa, ob, M, N, K, _pair(al), pA, lda, pB, ldb, None, 0,
                    _pair(0 if b0 else be), dC.ptr, M + pad)
            assert rc == 0
            bx.synchronize()
            out = dC.download()
            for d in (dA, dB, dC):
                d.free()
            assert np.array_equal(out, ref), (t, pad, off, shape, M, N, K, oa, ob)


@pytest.mark.parametrize("t,pad,off,shape", GIVEN)
def test_given_tile_triangles_integer_exact(gpu, t, pad, off, shape):
    """rank-k (and rank-2k) triangles on each compiled shape and movement: the
    stored triangle exact, the diagonal of a Hermitian update real, the other
    triangle untouched"""
    bx, dt = gpu, DT[t]
    fn, code = _tile_fn(bx), bx.dtype_code(dt)
    e, cplx = ROWS[shape], t == "Z"
    rng = np.random.default_rng(shape)
    m = 4 if t == "S" else 64
    for N, K in [(1, 20), (e - 1, 33), (e + 1, 8), (5 * e + 3, 40), (11 * e, 17)]:
        for j, (tri, opa) in enumerate([(1, 0), (2, 1), (2, 0), (1, 1)]):
            herm = cplx and j % 2 == 0
            two = j >= 2  # a second K segment: B op(A)^T
            say("given triangle", t, pad, off, shape, N, K, tri, opa, herm, two)
            oa = opa * (2 if herm else 1)
            ob = 0 if opa else (2 if herm else 1)
            sh = (K, N) if opa else (N, K)
            ld = _even(sh[0], dt, pad)
            A, B, C0 = (_ints(rng, dt, x, m) for x in ((ld, sh[1]), (ld, sh[1]), (N + pad, N)))
            X, Y = ((x[:sh[0]].T if opa else x[:sh[0]]) for x in (A, B))  # op(A) = X, or conj(X)
            tr = (lambda x: x.conj().T) if herm else (lambda x: x.T)
            if opa and herm:
                X, Y = X.conj(), Y.conj()
            al = 2.0 if herm or not cplx else 2 - 1j
            be = -1.0 if herm or not cplx else 1 + 3j
            full = al * (X @ tr(Y) + Y @ tr(X) if two else X @ tr(X)) + be * C0[:N]
            if herm:
                full[np.diag_indices(N)] = full[np.diag_indices(N)].real
            keep = np.tril(np.ones((N, N), bool)) if tri == 1 else np.triu(np.ones((N, N), bool))
            ref = C0.copy(order="F")
            ref[:N][keep] = full[keep]
            (dA, pA), (dB, pB) = _operand(bx, A, off), _operand(bx, B, off)
            dC = bx.DeviceArray.from_host(C0)
            rc = fn(code, shape, tri | (4 if herm else 0), oa, ob, N, N, K, _pair(al), pA, ld,
                    pB if two else pA, ld, pB if two else None, ld, _pair(be), dC.ptr, N + pad)
            assert rc == 0
            bx.synchronize()
            out = dC.download()
            for d in (dA, dB, dC):
                d.free()
            assert np.array_equal(out, ref), (t, pad, off, shape, N, K, tri, opa, herm, two)


@pytest.mark.parametrize("t", ["S", "D", "Z"])
def test_product_cut_into_launches_integer_exact(gpu, t):
    """what has more tiles than a launch may hold is cut into several: here at a
    few tiles, tall, wide and square, every transposition, with padding"""
    bx, dt = gpu, DT[t]
    fn, code = _tile_fn(bx), bx.dtype_code(dt)
    fn = bx.test_lib().bxtest_gemm_tile_most
    fn.argtypes = bx.test_lib().bxtest_gemm_tile.argtypes + [C.c_int64]
    cplx = t == "Z"
    op = (lambda x: x, lambda x: x.T, lambda x: x.conj().T)
    al, be = (2 - 1j, 1 + 3j) if cplx else (3.0, -2.0)
    rng = np.random.default_rng(5)
    for M, N, K, most in [(1000, 3, 20, 4), (5, 1100, 33, 3), (700, 650, 24, 7), (200, 130, 8, 1)]:
        for oa in range(3 if cplx else 2):
            for ob in range(3 if cplx else 2):
                say("cut product", t, M, N, K, most, oa, ob)
                sa, sb = ((M, K) if oa == 0 else (K, M)), ((K, N) if ob == 0 else (N, K))
                A, B, C0 = (_ints(rng, dt, (r + 4, c), 4) for r, c in (sa, sb, (M, N)))
                ref = C0.copy(order="F")
                ref[:M] = al * (op[oa](A[:sa[0]]) @ op[ob](B[:sb[0]])) + be * C0[:M]
                dA, dB, dC = (bx.DeviceArray.from_host(x) for x in (A, B, C0))
                rc = fn(code, -1, 0, oa, ob, M, N, K, _pair(al), dA.ptr, sa[0] + 4, dB.ptr,
                        sb[0] + 4, None, 0, _pair(be), dC.ptr, M + 4, most)
                assert rc == 0
                bx.synchronize()
                out = dC.download()
                for d in (dA, dB, dC):
                    d.free()
                assert np.array_equal(out, ref), (t, M, N, K, most, oa, ob)


def test_skinny_product_of_600_million_columns(gpu):
    """more columns than a grid of 32-column tiles holds"""
    bx, n = gpu, 600_000_000
    A = bx.DeviceArray.from_host(np.full((1, 1), 3, np.float32))
    B, Cd = bx.DeviceArray(1, n, np.float32), bx.DeviceArray(1, n, np.float32)
    B.fill_uniform(1, 1)
    say("skinny", n)
    bx.device_gemm("N", "N", 1, n, 1, 1.0, A.ptr, 1, B.ptr, 1, 0.0, Cd.ptr, 1, np.float32)
    bx.synchronize()
    assert np.array_equal(Cd.download(), np.float32(3) * B.download())
    for d in (A, B, Cd):
        d.free()
