"""The block tile shapes that single, rank-k and grouped products take, from
the library's own rules, without a GPU.  Shapes of a single product: 0 32x32,
1 64x32, 2 64x64, 3 128x64, 4 128x128; of a grouped one (BXH_SHAPE_*): 0
128x128, 1 128x64, 2 64x64, 3 32x32."""
import ctypes as C

import numpy as np
import pytest

DIMS = [(32, 32), (64, 32), (64, 64), (128, 64), (128, 128)]
LOWER, UPPER = 1, 2


@pytest.fixture(scope="module")
def L(bx):
    T = bx.test_lib()
    T.bxtest_tile_shape.argtypes = [C.c_int] * 5 + [C.c_int64]
    T.bxtest_tile_walk.argtypes = [C.c_int] * 4 + [C.c_void_p, C.c_int64]
    T.bxtest_tile_walk.restype = C.c_int64
    return T


def test_large_complex_products_take_the_large_tiles(bx, L):
    """4096^3 and up: 64x64 or 128x64 ran 5 to 10% faster than 64x32 at every
    size measured; triangles from 12288 (fewer tiles fit a band) on 128x64;
    small and skinny products spread over the CUs on the small tiles."""
    for n in (4096, 6144, 8192, 16384, 32768):
        for k in (512, 4096, n):
            assert L.bxtest_tile_shape(bx.Z, 1, 0, n, n, k) in (2, 3), (n, k)
    for n in (12288, 16384, 32768):
        for k in (4096, 16384):
            assert L.bxtest_tile_shape(bx.Z, 1, 1, n, n, k) == 3, (n, k)
    assert L.bxtest_tile_shape(bx.Z, 1, 0, 4096, 64, 4096) == 0
    assert L.bxtest_tile_shape(bx.Z, 1, 0, 256, 256, 256) == 0
    assert L.bxtest_tile_shape(bx.Z, 1, 0, 1500, 1000, 1200) == 1


def _shapes(bx, L, dt, probs, big=1):
    d = (bx.GemmDesc * len(probs))(*[
        bx.make_desc(dt, "N", "N", m, n, k, 1.0, 4096, m + m % 4, 4096, k + k % 4, 1.0, 4096, m)
        for m, n, k in probs])
    out, np_, tot = (C.c_int * len(probs))(), (C.c_int * 2)(), (C.c_int * 2)()
    n = L.bxtest_grouped_shapes(d, len(probs), bx.Z if dt == "complex128" else bx.D, big, out,
                                np_, tot)
    return list(out[:n]), list(np_), list(tot)


def test_grouped_complex_problems_fill_whole_rounds(bx, L):
    """128x64 tiles where they take one round of 512 and 64x64 tiles more than
    their 768 places, and for many tiles of long K; not with half of a tile
    empty, nor in a server batch"""
    dt = "complex128"
    assert _shapes(bx, L, dt, [(2048, 2048, 2048)]) == ([1], [0, 1], [0, 512])
    assert _shapes(bx, L, dt, [(512, 512, 512)] * 12)[1] == [12, 0]  # 768 tiles of 64x64
    assert _shapes(bx, L, dt, [(512, 512, 512)] * 13)[1] == [0, 13]
    assert _shapes(bx, L, dt, [(512, 512, 512)] * 16)[1] == [0, 16]
    assert _shapes(bx, L, dt, [(512, 512, 512)] * 17)[1] == [17, 0]
    assert _shapes(bx, L, dt, [(256, 8192, 4096)] * 32)[1] == [0, 32]
    assert _shapes(bx, L, dt, [(256, 8192, 4095)] * 32)[1] == [32, 0]
    assert _shapes(bx, L, dt, [(300, 3000, 700)] * 3)[1] == [3, 0]
    assert _shapes(bx, L, dt, [(64, 4096, 1024)] * 7)[1] == [7, 0]
    assert _shapes(bx, L, dt, [(2048, 2048, 2048)], big=0)[1] == [1, 0]
    s, np_, tot = _shapes(bx, L, dt, [(1024, 2048, 64), (30, 30, 100), (2048, 960, 900)])
    assert s == [3, 1, 1] and np_ == [1, 2] and tot == [1, 496], (s, np_, tot)


def test_complex_rounds_of_the_tile_runtime(bx, L):
    """one 2048^2 round: not 64x64, whose 1024 tiles begin an uneven round"""
    shape, form, grid = C.c_int(), C.c_int(), C.c_int()
    L.bxtest_round_tile(bx.Z, 2048, 0, 0, 2048, 2048, 2048, C.byref(shape), C.byref(form),
                        C.byref(grid))
    assert shape.value != 2
    L.bxtest_round_tile(bx.Z, 8192, 0, 0, 8192, 8192, 8192, C.byref(shape), C.byref(form),
                        C.byref(grid))
    assert (shape.value, grid.value) == (1, -1)


# every shape that a plain or rank-k launch can take, with a product and a
# triangle that takes it: (type, by DMA, shape, (M, N, K), (N, K))
REACHED = [
    ("S", 1, 0, (300, 300, 300), (300, 300)), ("S", 1, 1, (9080, 345, 3), (2497, 9)),
    ("S", 1, 2, (36433, 2809, 3), (17059, 8)), ("S", 1, 3, (64847, 51209, 18093), (50381, 51477)),
    ("S", 0, 0, (134, 20, 65224), (100, 42057)), ("S", 0, 1, (54692, 92, 8), (3837, 642)),
    ("S", 0, 2, (49665, 4309, 3), (19331, 36)),
    ("D", 1, 0, (2960, 1, 4151), (356, 5432)), ("D", 1, 1, (13508, 15, 262), (2668, 1)),
    ("D", 1, 2, (4555, 413, 978), (4099, 565)), ("D", 1, 3, (627, 16269, 665), (37183, 3)),
    ("D", 1, 4, (5304, 701, 14400), (63076, 53963)),
    ("D", 0, 0, (200, 4591, 941), (168, 4000)), ("D", 0, 1, (3784, 79, 260), (3061, 72)),
    ("D", 0, 2, (806, 3520, 777), (8886, 189)),
    ("Z", 1, 0, (211, 3000, 77), (200, 745)), ("Z", 1, 1, (10395, 25, 2677), (3601, 15)),
    ("Z", 1, 2, (13363, 36, 14823), (2651, 2011)), ("Z", 1, 3, (16384, 16384, 4096), (36851, 3)),
    ("Z", 0, 0, (725, 36, 67), (212, 2000)), ("Z", 0, 1, (11216, 31, 13726), (707, 11637)),
    ("Z", 0, 2, (2490, 2823, 259), (8645, 1)),
]


def test_shapes_taken_per_type(bx, L):
    """the shapes compiled for plain launches are those that the costs can
    pick: each is taken by some product and some triangle, and no other is"""
    code = {"S": bx.S, "D": bx.D, "Z": bx.Z}
    have = {"S1": 4, "S0": 3, "D1": 5, "D0": 3, "Z1": 4, "Z0": 3}
    assert {k: len({r[2] for r in REACHED if f"{r[0]}{r[1]}" == k}) for k in have} == have
    for t, dma, s, (m, n, k), (tn, tk) in REACHED:
        assert L.bxtest_tile_shape(code[t], dma, 0, m, n, k) == s, (t, dma, s)
        assert L.bxtest_tile_shape(code[t], dma, LOWER, tn, tn, tk) == s, (t, dma, s)
    rng = np.random.default_rng(1)
    for m, n, k in np.exp(rng.uniform(0, np.log(65536), (20000, 3))).astype(int) + 1:
        for t in code:
            for dma in (0, 1):
                for tri in (0, LOWER):
                    s = L.bxtest_tile_shape(code[t], dma, tri, m, m if tri else n, k)
                    assert s < have[f"{t}{dma}"], (t, dma, tri, m, n, k, s)


def _walk(L, shape, tri, m, n, cap=400000):
    buf = np.empty((cap, 2), np.int32)
    k = L.bxtest_tile_walk(shape, tri, m, n, buf.ctypes.data, cap)
    assert k >= 0
    return buf[:k]


@pytest.mark.parametrize("shape", range(5))
def test_triangle_walk_takes_each_tile_once(bx, L, shape):
    """every tile with an element on the stored triangle, once; the rest of the
    grid are tiles of the matrix beside the diagonal, each once too"""
    bm, bn = DIMS[shape]
    rng = np.random.default_rng(shape)
    for n in [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 1000, 1024, 2100,
              4000] + list(rng.integers(1, 5000, 12)):
        tm, tn = -(-n // bm), -(-n // bn)
        for tri in (LOWER, UPPER):
            got = _walk(L, shape, tri, n, n)
            seen = np.zeros((tm, tn), int)
            np.add.at(seen, (got[:, 0], got[:, 1]), 1)  # IndexError outside the matrix
            assert got.min() >= 0 and seen.max() == 1, (n, tri)
            r0, c0 = np.arange(tm) * bm, np.arange(tn) * bn
            r1, c1 = np.minimum(r0 + bm, n) - 1, np.minimum(c0 + bn, n) - 1
            need = (r1[:, None] >= c0) if tri == LOWER else (r0[:, None] <= c1)
            assert np.all(seen[need] == 1), (n, tri)


@pytest.mark.parametrize("m,n", [(1, 1), (500, 130), (129, 5000), (4097, 1000), (640, 640),
                                 (3000, 9000), (16384, 8192)])
def test_striped_walk_takes_each_tile_once(bx, L, m, n):
    got = _walk(L, 4, 0, m, n)
    tm, tn = -(-m // 128), -(-n // 128)
    assert len(got) == tm * tn
    assert np.array_equal(np.unique(got[:, 0] * tn + got[:, 1]), np.arange(tm * tn))


def test_tiles_of_a_launch_fit_its_grid(bx, L):
    """a launch of 256 threads a tile takes fewer than 2^24 tiles: long skinny
    products (all within a GPU's memory) take a larger tile where a small one
    would have more; only beyond the largest tile is a product cut"""
    code = {"S": bx.S, "D": bx.D, "Z": bx.Z}
    for t, dma, m, n, k in [("D", 1, 131, 162670080, 85), ("D", 1, 1, 600_000_000, 4),
                            ("S", 1, 67, 1044287977, 1), ("S", 1, 600_000_000, 1, 1),
                            ("S", 0, 64, 900_000_000, 2), ("D", 0, 65, 522693628, 2),
                            ("Z", 1, 1_000_000_000, 3, 1), ("Z", 0, 1_000_000_000, 3, 1)]:
        bm, bn = DIMS[L.bxtest_tile_shape(code[t], dma, 0, m, n, k)]
        assert -(-m // bm) * -(-n // bn) < 2**24, (t, dma, m, n, k)
    for t in code:
        bm, bn = DIMS[L.bxtest_tile_shape(code[t], 1, LOWER, 265264, 265264, 680)]
        assert -(-265264 // bm) * -(-265264 // bn) / 2 < 2**24
