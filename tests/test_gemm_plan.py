"""The GEMM planner's choices, which need no device: which f32 grads
share a launch, and when the two grads of a matmul may run on two streams."""
from __future__ import annotations

import ctypes as C

import pytest

import picograd_amd


@pytest.fixture(scope="module")
def k():
    lib = picograd_amd.load().lib
    sz, i = C.c_size_t, C.c_int
    lib.pgk_gemm16_plan.restype, lib.pgk_gemm16_plan.argtypes = i, [i, i, sz, sz, sz, sz, i, C.POINTER(i)]
    lib.pgm_grad_split.restype, lib.pgm_grad_split.argtypes = i, [sz] * 7 + [C.POINTER(C.c_bool)]
    return lib


@pytest.mark.parametrize("m,kk,n,tile", [(8192, 64, 64, 0), (16384, 64, 64, 0), (2048, 256, 256, 0), (752, 424, 66, 0),
                                         (45, 270, 985, 0), (437, 613, 56, 32), (711, 189, 1293, 32),
                                         (256, 784, 512, 32), (256, 256, 512, 16)])
def test_f32_pairs_decline_a_long_reduction_on_the_larger_tile(k, m, kk, n, tile):
    k.pgk_gemm_f32_pair_tile.restype, k.pgk_gemm_f32_pair_tile.argtypes = C.c_int, [C.c_size_t] * 3
    assert k.pgk_gemm_f32_pair_tile(m, n, kk) == tile


@pytest.mark.parametrize("M,K,N,B,two", [
    (30, 1208, 16, 1, False), (16, 1072, 16, 1, False), (118, 2275, 16, 1, False), (32, 1439, 48, 15, False),
    (512, 128, 512, 32, False),  # one launch holds both
    (4097, 1000, 3000, 1, True),  # tiled plans for both
])
def test_grads_of_a_few_microseconds_stay_on_one_stream(k, M, K, N, B, two):
    """A second stream's fork and join cost more than either product."""
    streams = C.c_bool(not two)
    k.pgm_grad_split(M, K, N, N, B, M, B, C.byref(streams))
    assert streams.value == two
