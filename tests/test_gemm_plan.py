"""The GEMM planner's choices, which need no device: when the two grads of a
matmul may run on two streams."""
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
