"""Which side runs a product by default (the plan is a pure function, so no GPU is needed): the ranges where
hipBLASLt measured faster go there, their neighbours stay with the library's own kernel, and so does
everything that kernel cannot load."""
import ctypes

import pytest

from qwen3_5_native import hip

CUS, WS = 256, 32 << 20


def plan(M, N, K, ldy=None, ws=WS, modelled=0, cus=CUS):
    tile, split = ctypes.c_int(), ctypes.c_int()
    hip.check(hip.load().q35_gemm_default_plan(M, N, K, ldy or N, ws, cus, modelled, tile, split), "plan")
    return tile.value, split.value


@pytest.mark.parametrize("M,N,K", [
    (1, 1024, 1024), (16, 6400, 1536), (2, 264, 384),      # few rows, short K in whole 128s
    (1, 5120, 6144), (16, 5120, 4608), (9, 8192, 8192),    # few rows, deep K in whole 512s
    (17, 1024, 1280), (400, 512, 1152), (30, 512, 1024),   # few weights in two to four parts
    (80, 12352, 2560), (128, 12352, 2560), (160, 12352, 2560),  # 64-row tiles, one round
    (144, 5120, 6144),                                     # 64 x 64 tiles over a deep K
    (24, 9784, 2816),                                      # many parts of few rows
    (4096, 8192, 8192), (4096, 4096, 4096), (2062, 14336, 5120),  # 256 x 256 tiles
    (1300, 8192, 11008),                                   # the other large tiles, one round
    (3000, 5120, 17408), (3000, 19456, 2560), (1100, 2560, 4096),  # the first rules
])
def test_where_hipblaslt_is_faster(M, N, K):
    assert plan(M, N, K)[0] == -1
    assert plan(M, N, K, modelled=1)[0] >= 0  # the own kernel could run it


@pytest.mark.parametrize("M,N,K", [
    (1, 1024, 1088), (1, 8192, 1024), (17, 5120, 6144), (1, 5120, 6208), (17, 1024, 3712), (256, 12352, 2560),
    (128, 19456, 2560), (333, 19456, 2560), (333, 2560, 9728), (1217, 34816, 5120), (1217, 5120, 17408),
    (4096, 12352, 2560), (250, 5120, 6144)])
def test_where_the_own_kernel_stays(M, N, K):
    assert plan(M, N, K)[0] >= 0
    assert plan(M, N, K) == plan(M, N, K, modelled=1)


@pytest.mark.parametrize("M,N,K,ldy", [(70, 136, 200, 136), (70, 132, 192, 132), (70, 136, 192, 140)])
def test_what_the_own_kernel_does_not_take(M, N, K, ldy):
    assert plan(M, N, K, ldy) == (-1, 1) and plan(M, N, K, ldy, modelled=1) == (-1, 1)


def test_splits_fit_the_workspace():
    assert plan(333, 2560, 9728)[1] > 1
    assert plan(333, 2560, 9728, ws=0)[1] == 1
    assert plan(333, 2560, 9728, cus=0) == (-1, 1)  # the device could not be read
