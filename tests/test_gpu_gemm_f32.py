"""The f32 GEMM kernels at the sizes where their tiles can go wrong.

Every element against the f64 product of the same operands, within the bound
of K rounded products and K rounded additions in any order,
(gamma(K) + u) sum |a b| with u = 2^-23 (gemm_check.gamma; f32 products round,
unlike 16-bit ones, hence K + 1 roundings per term), plus the addition of C
with beta.  C sits inside a buffer of sentinels that must survive.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gemm_check import gamma

pytestmark = pytest.mark.gpu

SENTINEL = np.float32(-3.0e33)


@pytest.fixture(scope="module")
def gemm(lib):
    f = lib.lib.pgk_gemm_f32
    sz, vp = C.c_size_t, C.c_void_p
    f.restype = C.c_int
    f.argtypes = [C.c_int, C.c_int, sz, sz, sz, vp, sz, sz, vp, sz, sz, vp, sz, sz, sz, C.c_int, vp]
    return f


# (m, n, k, batch): one 16-tile and its edges, reductions shorter than a wave's
# share, k not a multiple of 4, 8, 16 or 64; 1024 16-tiles, and 32-tiles past
# them; 64-tiles from 176 of them up; 128-tiles
SHAPES = [(1, 1, 1, 1), (1, 33, 7, 3), (31, 32, 64, 1), (33, 65, 513, 2), (10, 16, 2049, 1),
          (512, 509, 150, 1), (545, 515, 131, 1), (512, 544, 300, 1),
          (1025, 769, 64, 1), (1024, 1024, 63, 1), (1020, 772, 132, 2), (65, 64, 130, 130),
          (2944, 2945, 33, 1), (3072, 3072, 68, 1), (5, 9, 0, 2)]


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("shape", SHAPES)
def test_gemm_f32_every_element(lib, gemm, shape, ta, tb):
    m, n, k, b = shape
    rng = np.random.default_rng(m * 7 + n * 5 + k * 3 + b)
    # odd shapes with padded leading dims too (a 4-byte aligned operand), even ones dense
    pad = 3 if (m * n) % 2 else 0
    a = rng.standard_normal((b, k, m + pad) if ta else (b, m, k + pad)).astype(np.float32)
    w = rng.standard_normal((b, n, k + pad) if tb else (b, k, n + pad)).astype(np.float32)
    A = a[..., :m].swapaxes(1, 2) if ta else a[..., :k]
    W = w[..., :k].swapaxes(1, 2) if tb else w[..., :n]
    A64, W64 = A.astype(np.float64), W.astype(np.float64)
    ldc, rows = n + 5, m + 4
    c0 = np.full((b, rows, ldc), SENTINEL, np.float32)
    c0[:, 2:2 + m, :n] = rng.standard_normal((b, m, n))
    ta_, tw_, tc_ = lib.tensor(a.reshape(-1) if a.size else np.zeros(1, np.float32)), \
        lib.tensor(w.reshape(-1) if w.size else np.zeros(1, np.float32)), None
    ref, mag = A64 @ W64, np.abs(A64) @ np.abs(W64)
    for beta in (0, 1):
        tc_ = lib.tensor(c0.reshape(-1))
        st = lib.pg_amd_stream()
        rc = gemm(ta, tb, m, n, k, lib.tinfo(ta_).dev, a.shape[2], a[0].size, lib.tinfo(tw_).dev, w.shape[2], w[0].size,
                  lib.tinfo(tc_).dev + 4 * 2 * ldc, ldc, rows * ldc, b, beta, st)
        assert rc == 0
        got = lib.read(tc_).reshape(c0.shape)
        lib.pg_tensor_free(tc_)
        inner = got[:, 2:2 + m, :n].astype(np.float64)
        base = c0[:, 2:2 + m, :n].astype(np.float64) if beta else 0.0
        bound = gamma(k + 2) * (mag + np.abs(base)) + 1e-38
        bad = np.abs(inner - (ref + base)) > bound
        assert not bad.any(), (shape, ta, tb, beta, np.argwhere(bad)[:4].tolist())
        got[:, 2:2 + m, :n] = SENTINEL
        assert (got == SENTINEL).all()
    lib.pg_tensor_free(ta_)
    lib.pg_tensor_free(tw_)


def test_gemm_f32_special_values(lib, gemm):
    """Infinities and NaN reach their own row and column only, also at the
    edge of a tile and of k; subnormal products and operands are kept."""
    m, n, k = 70, 66, 37
    rng = np.random.default_rng(5)
    a = rng.standard_normal((m, k)).astype(np.float32)
    w = rng.standard_normal((k, n)).astype(np.float32)
    a[m - 1, k - 1], a[32, 3], w[k - 1, n - 1] = np.inf, np.nan, -np.inf
    a[5], w[:, 7] = 0.0, 0.0
    a[5, 0], w[0, 7] = np.float32(2.0 ** -70), np.float32(2.0 ** -70)   # product 2^-140
    a[6], w[:, 8] = 0.0, 0.0
    a[6, 1], w[1, 8] = np.float32(2.0 ** -140), np.float32(0.5)
    ta, tw, tc = lib.tensor(a), lib.tensor(w), lib.tensor(np.zeros((m, n), np.float32))
    st = lib.pg_amd_stream()
    assert gemm(0, 0, m, n, k, lib.tinfo(ta).dev, k, 0, lib.tinfo(tw).dev, n, 0, lib.tinfo(tc).dev, n, 0, 1, 0, st) == 0
    got = lib.read(tc)
    with np.errstate(all="ignore"):
        ref = a.astype(np.float64) @ w.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), fin)
    assert got[5, 7] == np.float32(2.0 ** -140) and got[6, 8] == np.float32(2.0 ** -141)
    for t in (ta, tw, tc):
        lib.pg_tensor_free(t)


@pytest.mark.parametrize("abat,bbat", [(1, 1), (1, 0), (0, 1)])
def test_matmul_f32_batched_backward(lib, abat, bbat):
    """Each batched form's grads, twice over one graph (a second pass overwrites)."""
    b, m, k, n = 3, 37, 29, 41
    rng = np.random.default_rng(9)
    a = rng.standard_normal((b, m, k) if abat else (m, k)).astype(np.float32)
    w = rng.standard_normal((b, k, n) if bbat else (k, n)).astype(np.float32)
    g = rng.standard_normal((b, m, n)).astype(np.float32)
    na, nw, tg = lib.var(a), lib.var(w), lib.tensor(g)
    y = lib.op("matmul", na, nw)
    for _ in range(2):
        lib.pg_amd_backward_from(y, tg)
        a64, w64, g64 = (x.astype(np.float64) for x in (a, w, g))
        da = g64 @ np.swapaxes(w64, -1, -2)
        dw = np.swapaxes(a64, -1, -2) @ g64
        da, dw = da if abat else da.sum(0), dw if bbat else dw.sum(0)
        for node, ref in ((na, da), (nw, dw)):
            got = lib.grad(node)
            assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
            assert np.abs(got - ref).max() <= 1e-4
    lib.pg_node_free(y)
    lib.pg_tensor_free(tg)
    lib.pg_node_free(na)
    lib.pg_node_free(nw)


# (m, k, n) around what one launch holds: 16-tiles up to 1024 of them in all,
# odd and even rows, more of them (32-tiles), and a pair that is too large
@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (17, 33, 10), (200, 20, 1001), (256, 256, 512), (260, 500, 300),
                                   (640, 784, 512), (1300, 1100, 65)])
@pytest.mark.parametrize("beta", [0, 1])
def test_matmul_f32_backward_pair(lib, gemm, m, k, n, beta):
    """Both grads of a product in one launch against f64, and against the two
    launches they replace; C of neither reaches past its own elements."""
    f = lib.lib.pgk_gemm_f32_pair
    sz, vp = C.c_size_t, C.c_void_p
    f.restype, f.argtypes = C.c_int, [sz, sz, sz, vp, vp, vp, vp, C.c_int, vp, C.c_int, vp]
    rng = np.random.default_rng(m + 3 * k + 5 * n)
    a, b, g = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    a64, b64, g64 = (x.astype(np.float64) for x in (a, b, g))
    ta, tb, tg = lib.tensor(a), lib.tensor(b), lib.tensor(g)
    pa, pb, pg = (lib.tinfo(t).dev for t in (ta, tb, tg))
    c0 = [np.full(r * c + 64, SENTINEL, np.float32) for r, c in ((m, k), (k, n))]
    for x, size in zip(c0, (m * k, k * n)):
        x[:size] = rng.standard_normal(size)
    one, two = [lib.tensor(x) for x in c0], [lib.tensor(x) for x in c0]
    st = lib.pg_amd_stream()
    rc = f(m, n, k, pa, pb, pg, lib.tinfo(one[0]).dev, beta, lib.tinfo(one[1]).dev, 1 - beta, st)
    assert rc == (-1 if m == 1300 else 0)
    assert gemm(0, 1, m, k, n, pg, n, 0, pb, n, 0, lib.tinfo(two[0]).dev, k, 0, 1, beta, st) == 0
    assert gemm(1, 0, k, n, m, pa, k, 0, pg, n, 0, lib.tinfo(two[1]).dev, n, 0, 1, 1 - beta, st) == 0
    refs = ((g64 @ b64.T, np.abs(g64) @ np.abs(b64.T), n, beta), (a64.T @ g64, np.abs(a64.T) @ np.abs(g64), m, 1 - beta))
    for t, t2, x, (ref, mag, red, bt) in zip(one, two, c0, refs):
        got, got2 = lib.read(t), lib.read(t2)
        size = ref.size
        if rc:
            assert np.array_equal(got, x)
            got = got2
        base = x[:size].astype(np.float64) * bt
        bound = gamma(red + 2) * (mag.reshape(-1) + np.abs(base)) + 1e-38
        for y in (got, got2):
            assert (np.abs(y[:size] - (ref.reshape(-1) + base)) <= bound).all()
            assert (y[size:] == SENTINEL).all()
    for t in (ta, tb, tg, *one, *two):
        lib.pg_tensor_free(t)


def test_matmul_f32_backward_shared_operand(lib):
    """x x has one grad, the sum of both products: never written side by side."""
    n = 96
    x = np.random.default_rng(3).standard_normal((n, n)).astype(np.float32)
    g = np.random.default_rng(4).standard_normal((n, n)).astype(np.float32)
    nx, tg = lib.var(x), lib.tensor(g)
    y = lib.op("matmul", nx, nx)
    x64, g64 = x.astype(np.float64), g.astype(np.float64)
    mag = np.abs(g64) @ np.abs(x64.T) + np.abs(x64.T) @ np.abs(g64)
    for _ in range(2):
        lib.pg_amd_backward_from(y, tg)
        assert (np.abs(lib.grad(nx) - (g64 @ x64.T + x64.T @ g64)) <= gamma(n + 3) * mag).all()
    lib.pg_node_free(y)
    lib.pg_tensor_free(tg)
    lib.pg_node_free(nx)
