"""The block tile shapes that single, rank-k and grouped products take, from
the library's own rules, without a GPU.  Shapes of a single product: 0 32x32,
1 64x32, 2 64x64, 3 128x64, 4 128x128; of a grouped one (BXH_SHAPE_*): 0
128x128, 1 128x64, 2 64x64, 3 32x32."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def L(bx):
    T = bx.test_lib()
    T.bxtest_tile_shape.argtypes = [C.c_int] * 5 + [C.c_int64]
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
