"""Which kernel a linear's sizes run on (the rules are host code: no GPU is
needed here).  Each row is a side of one of the rules' lines, measured."""

from __future__ import annotations

import ctypes

import pytest

STREAM, SKINNY, SLAB, GROUPED = range(4)


@pytest.fixture(scope="module")
def lib(built_lib):
    from ccut import _lib

    return _lib.lib()


@pytest.mark.parametrize("M,K,N,G,kernel", [
    (1, 4096, 14336, 128, STREAM), (16, 4096, 14336, 128, STREAM), (16, 4096, 14336, 64, SKINNY),
    (16, 4224, 14336, 128, SKINNY), (64, 4096, 4096, 128, SKINNY), (37, 4096, 14336, 128, SLAB),
    (2048, 4096, 14336, 64, SLAB), (2048, 4096, 14336, 128, GROUPED),
    # many rows of a short K: two rounds of 64 x 64 blocks, and past those
    (1024, 512, 2048, 128, SKINNY), (8192, 256, 512, 128, GROUPED), (1024, 512, 2176, 128, GROUPED),
    # where the 64-row kernel would be slower than the 16-row one, and just past
    (65, 2048, 8224, 128, SKINNY), (65, 2176, 8224, 128, SLAB), (96, 2048, 8224, 128, SLAB),
    (128, 1536, 8256, 32, SKINNY), (128, 1664, 8256, 32, SLAB), (128, 640, 8256, 32, SLAB),
    (2048, 256, 4096, 64, SKINNY), (2048, 384, 4096, 64, SLAB), (65, 256, 14336, 32, SKINNY), (96, 256, 14336, 32, SLAB),
    (2048, 1024, 4096, 64, SKINNY), (2048, 1152, 4096, 64, SLAB), (2048, 512, 4096, 64, SLAB), (2048, 1024, 4160, 64, SLAB),
    (128, 3072, 2048, 32, SKINNY), (64, 3072, 4096, 32, SKINNY), (64, 3072, 8192, 32, SLAB), (512, 3072, 1024, 64, SKINNY),
    (768, 3072, 512, 32, SKINNY), (121, 2176, 4096, 32, SLAB), (139, 2816, 2112, 32, SLAB),
    (0, 128, 16, 128, -1), (1, 64, 16, 128, -1), (1, 128, 8, 128, -1), (1, 128, 16, 16, -1),
])
def test_awq_linear(lib, M, K, N, G, kernel):
    assert lib.ccq_w4_gemm_kernel(M, K, N, G) == kernel


FP8_ROW, INT8_ROW, MXFP8, MXFP4 = range(4)


def wq(lib, fmt, M, K, N, G=32):
    """(kernel, rows, columns of a workgroup)"""
    r, c = ctypes.c_int(), ctypes.c_int()
    return lib.ccq_wq_linear_kernel(fmt, M, K, N, G, ctypes.byref(r), ctypes.byref(c)), r.value, c.value


@pytest.mark.parametrize("fmt,M,K,N,route", [
    (FP8_ROW, 512, 4096, 14336, (3, 128, 256)), (FP8_ROW, 500, 256, 10300, (3, 128, 256)),
    (FP8_ROW, 260, 256, 7000, (3, 128, 128)), (FP8_ROW, 260, 320, 7000, (3, 128, 128)),
    (FP8_ROW, 300, 768, 4100, (3, 64, 128)), (FP8_ROW, 16, 4096, 14336, (1, 16, 64)),
    (FP8_ROW, 16, 4096, 8192, (2, 16, 32)), (MXFP4, 16, 4096, 14336, (2, 16, 64)),
    # a short K stays on the 64-row kernel, by columns of a workgroup
    (FP8_ROW, 16, 256, 4096, (2, 16, 16)), (FP8_ROW, 16, 1792, 4100, (1, 16, 64)), (INT8_ROW, 4, 1024, 8192, (1, 16, 64)),
    (FP8_ROW, 16, 2048, 8192, (2, 16, 32)), (MXFP8, 1, 256, 33, (1, 16, 64)), (MXFP8, 1, 512, 33, (2, 16, 16)),
    (MXFP8, 16, 1280, 8192, (1, 16, 64)), (MXFP8, 16, 1536, 8192, (2, 16, 32)), (MXFP4, 16, 256, 8192, (1, 16, 64)),
    (MXFP4, 16, 512, 8192, (2, 16, 32)), (MXFP4, 1, 3072, 14336, (1, 16, 64)), (MXFP4, 1, 3328, 14336, (2, 16, 64)),
    # in_features % 256 != 0: rows times columns from which the tiles are faster
    (INT8_ROW, 48, 1600, 4096, (3, 64, 128)), (INT8_ROW, 48, 2112, 4096, (0, 0, 0)), (INT8_ROW, 49, 2112, 4096, (3, 64, 128)),
    (INT8_ROW, 51, 4224, 4096, (0, 0, 0)), (INT8_ROW, 56, 4224, 4096, (3, 64, 128)), (FP8_ROW, 49, 4224, 4096, (3, 64, 128)),
    (MXFP8, 32, 1088, 4096, (3, 64, 128)), (MXFP8, 32, 2176, 4096, (0, 0, 0)), (MXFP8, 36, 2176, 4096, (3, 64, 128)),
    (MXFP8, 48, 4224, 4096, (0, 0, 0)), (MXFP8, 49, 4224, 4096, (3, 64, 128)), (MXFP4, 32, 4224, 4096, (3, 64, 128)),
    (MXFP4, 64, 4096, 14336, (1, 64, 64)), (MXFP4, 12, 4224, 14336, (0, 0, 0)),
])
def test_decoded_weight_linear(lib, fmt, M, K, N, route):
    assert wq(lib, fmt, M, K, N) == route


@pytest.mark.parametrize("fmt,M,K,N,route", [
    (MXFP4, 16, 512, 8192, (1, 16, 64)), (MXFP4, 16, 768, 8192, (2, 16, 32)), (MXFP4, 16, 2048, 14336, (2, 16, 64)),
    (MXFP4, 16, 2304, 14336, (1, 16, 64)), (MXFP4, 16, 4096, 14336, (2, 16, 64)), (MXFP4, 16, 4352, 14336, (1, 16, 64)),
    (MXFP4, 16, 5120, 14336, (2, 16, 64)), (MXFP8, 16, 512, 8192, (1, 16, 64)),
])
def test_decoded_weight_linear_groups_of_16(lib, fmt, M, K, N, route):
    assert wq(lib, fmt, M, K, N, 16) == route


@pytest.mark.parametrize("M,K,N,kernel", [
    (32, 4096, 4096, 1), (1024, 4096, 4096, 2), (4096, 4096, 14336, 3), (1024, 4112, 4096, 4), (40, 20, 100, 0),
    # rounds of the CUs with 256- and with 128-row tiles: 3 and 5, 2 and 3, 1 and 2
    (4096, 1024, 5120, 3), (257, 512, 28672, 2), (1536, 4096, 8192, 2), (260, 1280, 16500, 2), (260, 1280, 16300, 3),
])
def test_int8_linear(lib, M, K, N, kernel):
    assert lib.ccq_int8_linear_kernel(M, K, N) == kernel
