"""The GEMM planner's choices, which need no device: which products take the
tiles whose waves split the reduction (planner tiles 5 to 8) and the few-rows
kernel (9), alone and as a dgrad + wgrad pair, which f32 grads share a launch,
and when the two grads of a matmul may run on two streams."""
from __future__ import annotations

import ctypes as C

import pytest

import picograd_amd
from test_gpu_gemm_guard import GemmDesc


@pytest.fixture(scope="module")
def k():
    lib = picograd_amd.load().lib
    sz, i = C.c_size_t, C.c_int
    lib.pgk_gemm16_plan.restype, lib.pgk_gemm16_plan.argtypes = i, [i, i, sz, sz, sz, sz, i, C.POINTER(i)]
    lib.pgk_gemm16_ks_pair_tile.restype = i
    lib.pgk_gemm16_ks_pair_tile.argtypes = [C.POINTER(GemmDesc), C.POINTER(GemmDesc)]
    lib.pgm_grad_split.restype, lib.pgm_grad_split.argtypes = i, [sz] * 7 + [C.POINTER(C.c_bool)]
    return lib


def pair_tile(k, M, K, N):
    """For dX [M, K] = G W^T and dW [K, N] = X^T G."""
    d = GemmDesc(M, K, N, 16, N, 0, M, 16, N, 0, K, 16, K, 0, 1, 0)
    w = GemmDesc(K, N, M, 16, K, 0, K, 16, N, 0, N, 16, N, 0, 1, 0)
    return k.pgk_gemm16_ks_pair_tile(C.byref(d), C.byref(w))


@pytest.mark.parametrize("m,n,kk,tile", [
    (512, 512, 4096, 5), (512, 512, 65536, 0), (64, 64, 16384, 0), (72, 1080, 7520, 0),
    (512, 1024, 4096, 6), (512, 1024, 16384, 0), (1024, 1024, 4096, 8), (1024, 1024, 16384, 0),
    (2048, 1024, 2048, 7), (2048, 1024, 12288, 0), (440, 3440, 5080, 0), (2232, 528, 2888, 0), (45, 3592, 3768, 5),
])
def test_long_reductions_keep_the_split_over_blocks(k, m, n, kk, tile):
    """A tile of one CU is taken up to the reduction at which eight slices of
    the chip are faster; 0 here is any of the tiled plans."""
    got = k.pgk_gemm16_plan(1, 1, m, n, kk, 1, 0, None)
    assert got == tile if tile else got in (1, 2, 3)


@pytest.mark.parametrize("ta,tb,kk,tile", [(1, 1, 6144, 5), (1, 1, 6152, 0), (0, 1, 10240, 5), (0, 0, 10240, 5), (0, 0, 10248, 0)])
def test_layouts_that_read_whole_lines_hold_further(k, ta, tb, kk, tile):
    got = k.pgk_gemm16_plan(ta, tb, 64, 640, kk, 1, 0, None)
    assert got == tile if tile else got in (1, 2, 3)


@pytest.mark.parametrize("m,n,kk,few", [(16, 4096, 4096, True), (16, 128, 8192, True), (64, 16, 32768, True),
                                        (5, 3232, 6192, True), (13, 64, 18896, False), (16, 3376, 25800, False)])
def test_few_rows_up_to_the_measured_reductions(k, m, n, kk, few):
    assert (k.pgk_gemm16_plan(0, 1, m, n, kk, 1, 0, None) == 9) == few


@pytest.mark.parametrize("M,K,N,tile", [
    (8192, 128, 1024, 0), (16384, 64, 512, 0), (16384, 64, 2048, 0), (8192, 64, 64, 0), (16384, 64, 64, 0),
    (4096, 64, 1024, 6), (4096, 256, 2048, 7), (7080, 32, 24, 5), (6928, 16, 88, 5), (5056, 80, 32, 8),
])
def test_pairs_look_at_the_longer_reduction(k, M, K, N, tile):
    assert pair_tile(k, M, K, N) == tile


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
