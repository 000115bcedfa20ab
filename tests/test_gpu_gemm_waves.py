"""The 16-bit GEMM tiles whose waves split the reduction (planner tiles 5 to
8), at the sizes where they can go wrong: one element, tile edges, a
reduction shorter than one wave's chunk, shorter than the eight waves'
chunks, ending mid-chunk, and the largest outputs each tile takes.

Every element against the f64 product within the f32 summation bound
(gemm_check), into a C placed between sentinels, with beta 0 and 1; the same
for a dgrad + wgrad pair in one launch, batched problems and the fused
epilogue of a linear16 layer.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gemm_check import check_linear, check_product
from picograd_amd.capi import BF16, F16
from test_gpu_gemm_guard import GUARD, Dev, GemmDesc, _c_buffer, _check_guards, _f32, _operands, k  # noqa: F401

pytestmark = pytest.mark.gpu

# (tile, m, n, k)
SHAPES = [
    (5, 17, 17, 8), (5, 31, 33, 24), (5, 33, 40, 64), (5, 64, 512, 513), (5, 256, 1024, 520), (5, 250, 1023, 40),
    (6, 512, 1024, 256), (6, 510, 1021, 264), (6, 17, 16384, 32), (6, 288, 1000, 8),
    (7, 1024, 1024, 72), (7, 1023, 2047, 136), (7, 2048, 1024, 16), (7, 600, 1000, 1000),
    (8, 600, 1000, 1024), (8, 1024, 1023, 1100),
]


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("lay", [(0, 0), (0, 1), (1, 0), (1, 1)], ids=["kk", "kn", "mk", "mn"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "t%d-%dx%dx%d" % s)
def test_split_over_waves(lib, oracle, k, shape, lay, dt):  # noqa: F811
    tile, m, n, kk = shape
    ta, tb = lay
    if not (ta and tb):
        kk = (kk + 7) // 8 * 8  # a K-contiguous operand's whole chunks
    beta = (m + n + dt) % 2
    what = f"gemm tile {tile} dt={dt} ta={ta} tb={tb} {m}x{n}x{kk} beta={beta}"
    print(what, flush=True)
    sp = C.c_int(0)
    assert k.pgk_gemm16_plan(ta, tb, m, n, kk, 1, 0, C.byref(sp)) == tile and sp.value == 1
    assert k.pgk_gemm16_workspace_cu(ta, tb, m, n, kk, 1, 0) == 0
    rng = np.random.default_rng(m * 31 + n * 7 + kk)
    A, B, a_st, lda, a_ext, b_st, ldb, b_ext = _operands(oracle, rng, dt, ta, tb, m, n, kk)
    buf, ldc, c0 = _c_buffer(rng, m, n, beta)
    d = Dev(k)
    try:
        pa, pb, pc = d.put(a_st), d.put(b_st), d.put(buf)
        rc = k.pgk_gemm16_cu(dt, ta, tb, m, n, kk, pa, lda, 0, a_ext, pb, ldb, 0, b_ext, pc + GUARD * ldc * 4, ldc,
                             0, 1, beta, None, None, 0, k.pgd_stream())
        assert rc == 0, rc
        after = d.get(pc, buf.shape, np.float32)
    finally:
        d.free()
    _check_guards(after, m, n, what)
    check_product(after[GUARD:GUARD + m, :n], [(_f32(dt, A), _f32(dt, B))], what, add=c0)


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("beta", [0, 1])
@pytest.mark.parametrize("m,n,kk", [(1, 1, 8), (1, 4096, 1024), (15, 17, 72), (16, 4095, 520), (5, 10, 4096), (64, 16, 584),
                                    (49, 7, 64), (16, 128, 8192)])
def test_few_rows(lib, oracle, k, m, n, kk, beta, dt):  # noqa: F811
    what = f"few rows dt={dt} {m}x{n}x{kk} beta={beta}"
    print(what, flush=True)
    sp = C.c_int(0)
    assert k.pgk_gemm16_plan(0, 1, m, n, kk, 1, 0, C.byref(sp)) == 9 and sp.value == 1
    assert k.pgk_gemm16_workspace_cu(0, 1, m, n, kk, 1, 0) == 0
    rng = np.random.default_rng(m * 31 + n * 7 + kk)
    A, B, a_st, lda, a_ext, b_st, ldb, b_ext = _operands(oracle, rng, dt, 0, 1, m, n, kk)
    buf, ldc, c0 = _c_buffer(rng, m, n, beta)
    d = Dev(k)
    try:
        pa, pb, pc = d.put(a_st), d.put(b_st), d.put(buf)
        rc = k.pgk_gemm16_cu(dt, 0, 1, m, n, kk, pa, lda, 0, a_ext, pb, ldb, 0, b_ext, pc + GUARD * ldc * 4, ldc,
                             0, 1, beta, None, None, 0, k.pgd_stream())
        assert rc == 0, rc
        after = d.get(pc, buf.shape, np.float32)
    finally:
        d.free()
    _check_guards(after, m, n, what)
    check_product(after[GUARD:GUARD + m, :n], [(_f32(dt, A), _f32(dt, B))], what, add=c0)


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("shape", [(40, 72, 104), (257, 264, 520), (130, 512, 1024), (1030, 264, 520), (500, 1000, 520), (96, 208, 616),
                                   (8160, 24, 32), (32, 32, 8192), (7160, 72, 72), (4096, 256, 200)],
                         ids=lambda s: "%dx%dx%d" % s)
def test_pair_in_one_launch(lib, oracle, k, shape, dt):  # noqa: F811
    """dX = G.W^T and dW = X^T.G of C = X.W, X [M, K], W [K, N]; dW accumulates."""
    M, K, N = shape
    what = f"waves pair dt={dt} M={M} K={K} N={N}"
    print(what, flush=True)
    rng = np.random.default_rng(M + N + dt)
    X = oracle.cast16(dt, rng.standard_normal((M, K)).astype(np.float32))
    W = oracle.cast16(dt, (0.05 * rng.standard_normal((K, N))).astype(np.float32))
    G = oracle.cast16(dt, rng.standard_normal((M, N)).astype(np.float32))
    bx, ldx, _ = _c_buffer(rng, M, K, 0)
    bw, ldw, c0w = _c_buffer(rng, K, N, 1)
    fn = k.pgk_gemm16_ks_pair
    fn.restype, fn.argtypes = C.c_int, [C.c_int, C.POINTER(GemmDesc), C.POINTER(GemmDesc), C.c_void_p]
    k.pgk_gemm16_ks_pair_tile.restype = C.c_int
    k.pgk_gemm16_ks_pair_tile.argtypes = [C.POINTER(GemmDesc), C.POINTER(GemmDesc)]
    d = Dev(k)
    try:
        pg, pw, px = d.put(G), d.put(W), d.put(X)
        cx, cw = d.put(bx), d.put(bw)
        dd = GemmDesc(M, K, N, pg, N, 0, M, pw, N, 0, K, cx + GUARD * ldx * 4, ldx, 0, 1, 0)
        dwd = GemmDesc(K, N, M, px, K, 0, K, pg, N, 0, N, cw + GUARD * ldw * 4, ldw, 0, 1, 1)
        assert k.pgk_gemm16_ks_pair_tile(C.byref(dd), C.byref(dwd)) in (5, 6, 7, 8)
        assert fn(dt, C.byref(dd), C.byref(dwd), k.pgd_stream()) == 0
        ax = d.get(cx, bx.shape, np.float32)
        aw = d.get(cw, bw.shape, np.float32)
    finally:
        d.free()
    _check_guards(ax, M, K, what + " dX")
    _check_guards(aw, K, N, what + " dW")
    f = lambda h: _f32(dt, h)  # noqa: E731
    check_product(ax[GUARD:GUARD + M, :K], [(f(G), f(W).T)], what + " dX")
    check_product(aw[GUARD:GUARD + K, :N], [(f(X).T, f(G))], what + " dW", add=c0w)


@pytest.mark.parametrize("M,K,N", [(2048, 512, 512), (4096, 256, 200), (560, 488, 3312)])
def test_pair_error_is_no_larger_than_the_split(lib, oracle, k, M, K, N):
    """Each grad's error against f64 beside that of the plan that splits the
    reduction over blocks (a budget of 255 CUs asks for a tiled plan): no fewer
    partial sums.  The two errors are norms over at least 51200 independent
    elements, so they differ by well under 5 % where the sums are alike; one sum
    per wave measures 1.2 to 1.4 times the split's."""
    print(f"pair error M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(M)
    X, W, G = (oracle.cast16(BF16, rng.standard_normal(s).astype(np.float32)) for s in ((M, K), (K, N), (M, N)))
    f = lambda h: _f32(BF16, h).astype(np.float64)  # noqa: E731
    refs = f(G) @ f(W).T, f(X).T @ f(G)
    fn = k.pgk_gemm16_ks_pair
    fn.restype, fn.argtypes = C.c_int, [C.c_int, C.POINTER(GemmDesc), C.POINTER(GemmDesc), C.c_void_p]
    d = Dev(k)
    try:
        pg, pw, px = d.put(G), d.put(W), d.put(X)
        cx, cw = d.put(np.zeros((M, K), np.float32)), d.put(np.zeros((K, N), np.float32))
        dd = GemmDesc(M, K, N, pg, N, 0, M, pw, N, 0, K, cx, K, 0, 1, 0)
        dwd = GemmDesc(K, N, M, px, K, 0, K, pg, N, 0, N, cw, N, 0, 1, 0)
        assert fn(BF16, C.byref(dd), C.byref(dwd), k.pgd_stream()) == 0
        pair = d.get(cx, (M, K), np.float32), d.get(cw, (K, N), np.float32)
        for ta, x in ((0, dd), (1, dwd)):
            wsz = k.pgk_gemm16_workspace_cu(ta, ta, x.m, x.n, x.k, 1, 255)
            ws = d.put(np.zeros(max(wsz, 16), np.uint8))
            assert k.pgk_gemm16_plan(ta, ta, x.m, x.n, x.k, 1, 255, None) < 5
            assert k.pgk_gemm16_cu(BF16, ta, ta, x.m, x.n, x.k, x.a, x.lda, 0, x.a_extent, x.b, x.ldb, 0, x.b_extent,
                                   x.c, x.ldc, 0, 1, 0, None, ws, 255, k.pgd_stream()) == 0
        split = d.get(cx, (M, K), np.float32), d.get(cw, (K, N), np.float32)
    finally:
        d.free()
    for name, got, ref, old in zip(("dX", "dW"), pair, refs, split):
        e, eo = np.linalg.norm(got - ref), np.linalg.norm(old - ref)
        assert e <= 1.05 * eo, (name, e / np.linalg.norm(ref), eo / np.linalg.norm(ref))


def test_missing_workspace_is_refused_before_anything_is_queued(lib, oracle, k):
    """A reduction with a tail (k % 8) on a tile of this file needs a workspace."""
    m, n, kk = 40, 48, 77
    rng = np.random.default_rng(1)
    A, B = (oracle.cast16(BF16, rng.standard_normal(s).astype(np.float32)) for s in ((m, 80), (n, 80)))
    c0 = rng.standard_normal((m, n)).astype(np.float32)
    assert k.pgk_gemm16_plan(0, 0, m, n, kk, 1, 0, None) == 5 and k.pgk_gemm16_workspace_cu(0, 0, m, n, kk, 1, 0)
    d = Dev(k)
    try:
        pa, pb, pc = d.put(A), d.put(B), d.put(c0)
        assert k.pgk_gemm16_cu(BF16, 0, 0, m, n, kk, pa, 80, 0, m, pb, 80, 0, n, pc, n, 0, 1, 0, None, None, 0,
                               k.pgd_stream()) != 0
        assert np.array_equal(d.get(pc, c0.shape, np.float32), c0)
    finally:
        d.free()


@pytest.mark.parametrize("M,K,N", [(30, 1202, 10), (118, 2275, 11)])
def test_matmul_with_small_grads(lib, oracle, M, K, N):
    """Grads that no one launch holds and that run one after the other."""
    print(f"waves matmul {M}x{K}x{N}", flush=True)
    rng = np.random.default_rng(M)
    a = oracle.cast16(F16, rng.standard_normal((M, K)).astype(np.float32))
    b = oracle.cast16(F16, rng.standard_normal((K, N)).astype(np.float32))
    g = _f32(F16, oracle.cast16(F16, rng.standard_normal((M, N)).astype(np.float32)))
    na, nb, tg = lib.var(a, dtype=F16), lib.var(b, dtype=F16), lib.tensor(g)
    y = lib.op("matmul", na, nb)
    lib.pg_amd_backward_from(y, tg)
    fa, fb = _f32(F16, a), _f32(F16, b)
    check_product(lib.value(y), [(fa, fb)], "forward")
    check_product(lib.grad(na), [(g, fb.T)], "dA")
    check_product(lib.grad(nb), [(fa.T, g)], "dB")
    lib.pg_node_free(y)
    lib.pg_tensor_free(tg)
    lib.pg_node_free(na)
    lib.pg_node_free(nb)


@pytest.mark.parametrize("batch,M,K,N", [(3, 65, 24, 40), (2, 200, 72, 136), (24, 64, 64, 128), (15, 32, 1439, 47)])
def test_batched_matmul(lib, oracle, batch, M, K, N):
    """pg_ag_matmul over batches: forward and both grads, each entry's own."""
    dt = F16
    print(f"waves bmm {batch}x{M}x{K}x{N}", flush=True)
    rng = np.random.default_rng(batch)
    a = oracle.cast16(dt, rng.standard_normal((batch, M, K)).astype(np.float32))
    b = oracle.cast16(dt, rng.standard_normal((batch, K, N)).astype(np.float32))
    g = _f32(dt, oracle.cast16(dt, rng.standard_normal((batch, M, N)).astype(np.float32)))
    na, nb, tg = lib.var(a, dtype=dt), lib.var(b, dtype=dt), lib.tensor(g)
    y = lib.op("matmul", na, nb)
    lib.pg_amd_backward_from(y, tg)
    fa, fb = _f32(dt, a), _f32(dt, b)
    check_product(lib.value(y), [(fa, fb)], "forward")
    check_product(lib.grad(na), [(g, np.swapaxes(fb, 1, 2))], "dA")
    check_product(lib.grad(nb), [(np.swapaxes(fa, 1, 2), g)], "dB")
    lib.pg_node_free(y)
    lib.pg_tensor_free(tg)
    lib.pg_node_free(na)
    lib.pg_node_free(nb)


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("M,K,N", [(5, 40, 24), (33, 64, 65), (300, 520, 1000), (1000, 136, 1048)])
def test_linear16_epilogue(lib, oracle, M, K, N, act, dt):
    print(f"waves linear16 act={act} dt={dt} {M}x{K}x{N}", flush=True)
    rng = np.random.default_rng(80 + dt + act)
    x = rng.standard_normal((M, K)).astype(np.float32)
    wt = (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
    b = (0.3 * rng.standard_normal(N)).astype(np.float32)
    nx, nw, nb = lib.var(x), lib.var(wt), lib.var(b)
    qx, qw = _f32(dt, oracle.cast16(dt, x)), _f32(dt, oracle.cast16(dt, wt))
    out = lib._check(lib.pg_amd_ag_linear16(nx, nw, nb, act, dt))
    z = lib.read(lib.pg_amd_linear16_preact(out)) if act else None
    check_linear(lib.value(out), z, [(qx, qw)], b, act, "layer")
    lib.pg_no_grad_push()
    out2 = lib._check(lib.pg_amd_ag_linear16(nx, nw, nb, act, dt))
    lib.pg_no_grad_pop()
    assert np.array_equal(lib.value(out2), lib.value(out))  # written by the epilogue, and formed from z
    for n in (out, out2, nx, nw, nb):
        lib.pg_node_free(n)
