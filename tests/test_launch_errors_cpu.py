"""A GEMM launch that fails reports HIP's own error through bxh_last_error:
launches without a device, on the CPU."""
import ctypes as C

import pytest

WHY = b"no ROCm-capable device"


@pytest.fixture(scope="module")
def L(bx):
    if bx.gpu_available():
        pytest.skip("needs a machine without a GPU")
    T = bx.test_lib()
    vp, i64 = C.c_void_p, C.c_int64
    T.bxtest_gemm_tile.argtypes = [C.c_int] * 8 + [vp, vp, i64, vp, i64, vp, i64, vp, vp, i64]
    T.bxtest_last_error.restype = C.c_char_p
    return T


@pytest.mark.parametrize("tri,what", [(0, b"gemm launch"), (1, b"rank-k launch")])
def test_single_launch_keeps_the_hip_error_cpu(bx, L, tri, what):
    one = (C.c_double * 2)(1.0, 0.0)
    for dt in (bx.S, bx.D, bx.Z):
        rc = L.bxtest_gemm_tile(dt, -1, tri, 0, 1, 64, 64, 64, one, 4096, 64, 4096, 64, None, 0,
                                one, 4096, 64)
        assert rc == -4 and what in L.bxtest_last_error() and WHY in L.bxtest_last_error()


def test_grouped_launch_keeps_the_hip_error_cpu(bx, L):
    for dt in (bx.S, bx.D, bx.Z):
        for grid in (0, -1):
            assert L.bxtest_gemm_grouped(dt, grid) == -4
            err = L.bxtest_last_error()
            assert b"grouped gemm launch" in err and WHY in err
    assert L.bxtest_gemm_grouped(7, 0) == -2
