"""Block tile shapes and operand movements of the plain device GEMM.

Integer inputs whose every partial sum is exact in the element type, so the
result must equal the naive oracle bit for bit at each tile's edges, at every
remainder of K, and for each way the operands are moved: 16-byte aligned,
element aligned (odd leading dimension, offset base), and with fewer rows
than one 16-byte load takes.
"""
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
# and longer, grids that pick each shape
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
    """a grid that takes the 128 x 64 tile, ragged in both dimensions"""
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
