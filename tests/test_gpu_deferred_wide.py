"""Forward runs above the one-block size: their sum_all and the backward
region join the run's main kernel.

Each shape goes where the tiling can go wrong: just above the one-block size,
few columns (row lanes in place of idle column lanes), columns that do not
divide by 4 or fill a 128-byte line, two rows, two columns.  The JIT path is
held to the eager path and to f64.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
from scipy.special import erf

pytestmark = pytest.mark.gpu

SHAPES = [(129, 128), (300, 100), (4097, 10), (9000, 2), (2, 8200), (515, 1037), (700, 260), (66, 4096)]


def launches(lib, f):
    """JIT main kernels (kind 0) that f launches."""
    lib.pg_amd_timer_reset()
    lib.pg_amd_timer_enable(1)
    f()
    lib.pg_amd_stream()
    cnt = C.c_size_t(0)
    lib.pg_amd_timer_read(0, C.byref(cnt))
    lib.pg_amd_timer_enable(0)
    lib.pg_amd_timer_reset()
    return cnt.value


def gate(lib, x, b, g, mean, passes=1):
    """gelu(x + b) * sigmoid(g), its sum (or picograd's mean_all) and grads."""
    nx, nb, ng = lib.var(x), lib.var(b), lib.var(g)
    lib.pg_amd_stream()
    out, made = {}, []

    def body():
        t0 = lib.op("add", nx, nb)
        t1 = lib.op("gelu", t0)
        t2 = lib.op("sigmoid", ng)
        y = lib.op("mul", t1, t2)
        loss = lib.op("mean_all" if mean else "sum_all", y)
        for _ in range(passes):
            lib.pg_backward(loss)
        made.extend([t0, t1, t2, y, loss])

    out["launches"] = launches(lib, body)
    for k, n in zip(("t0", "t1", "t2", "y", "loss"), made):
        out[k] = lib.value(n)
    for k, n in (("dx", nx), ("db", nb), ("dg", ng)):
        out[k] = lib.grad(n)
    for n in reversed(made):
        lib.pg_node_free(n)
    for n in (nx, nb, ng):
        lib.pg_node_free(n)
    return out


def f64_gate(x, b, g, mean):
    x, b, g = (v.astype(np.float64) for v in (x, b, g))
    z, s = x + b, 1 / (1 + np.exp(-g))
    phi = 0.5 * (1 + erf(z / np.sqrt(2)))
    sc = 1 / x.shape[1] if mean else 1.0
    dx = sc * s * (phi + z * np.exp(-0.5 * z * z) / np.sqrt(2 * np.pi))
    return {"y": z * phi * s, "loss": np.array([sc * (z * phi * s).sum()]), "dx": dx, "db": dx.sum(0),
            "dg": sc * z * phi * s * (1 - s)}


@pytest.mark.parametrize("mean", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_run_sum_and_backward_in_one_kernel(lib, shape, mean):
    rng = np.random.default_rng(shape[0] * 3 + shape[1])
    x, g = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    b = (0.1 * rng.standard_normal(shape[1])).astype(np.float32)
    got = {}
    for jit in (True, False):
        lib.pg_autograd_set_jit(jit)
        try:
            got[jit] = gate(lib, x, b, g, mean)
        finally:
            lib.pg_autograd_set_jit(True)
    assert got[True]["launches"] == 1
    ref = f64_gate(x, b, g, mean)
    for k in ("t0", "t1", "t2", "y"):  # uncontracted in the merged kernel: the eager kernels' bits
        assert np.array_equal(got[True][k].view(np.uint32), got[False][k].view(np.uint32)), k
    # the sums: rows + columns rounded additions of positive and negative terms
    u = 2.0 ** -24
    dep = (sum(shape) + 16) * u
    assert np.abs(got[True]["loss"] - ref["loss"]).max() <= 2 * dep * np.abs(ref["y"]).sum() / (shape[1] if mean else 1)
    assert (np.abs(got[True]["db"] - ref["db"]) <= (shape[0] + 16) * u * np.abs(ref["dx"]).sum(0) + 1e-6 *
            np.abs(ref["dx"]).max()).all()
    for k in ("dx", "dg"):
        scale = np.abs(ref[k]).max()
        assert np.abs(got[True][k] - ref[k]).max() <= 1e-6 * scale
        assert np.abs(got[True][k] - got[False][k]).max() <= 1e-6 * scale


def test_second_backward_overwrites(lib):
    """The second pass finds no pending run: the same grads from the region alone."""
    rng = np.random.default_rng(3)
    x, g = (rng.standard_normal((515, 1037)).astype(np.float32) for _ in range(2))
    b = rng.standard_normal(1037).astype(np.float32)
    one, two = gate(lib, x, b, g, False), gate(lib, x, b, g, False, passes=2)
    for k in ("dx", "db", "dg"):
        assert np.abs(one[k] - two[k]).max() <= 1e-6 * np.abs(one[k]).max() * (30 if k == "db" else 1)


def test_sum_without_backward(lib):
    """The recorded sum alone, then the output read, and a run whose sum is taken twice."""
    rng = np.random.default_rng(4)
    x = rng.standard_normal((777, 90)).astype(np.float32)
    nx = lib.var(x)
    y = lib.op("tanh", nx)
    s1 = lib.op("sum_all", y)
    s2 = lib.op("mean_all", y)
    want = np.tanh(x.astype(np.float64))
    assert np.abs(lib.value(y) - want).max() <= 1e-6
    assert abs(lib.value(s1)[0] - want.sum()) <= 1e-6 * np.abs(want).sum()
    assert abs(lib.value(s2)[0] - want.sum() / 90) <= 1e-6 * np.abs(want).sum() / 90
    for n in (s2, s1, y, nx):
        lib.pg_node_free(n)


def test_grads_summed_over_other_dims_stay_apart(lib):
    """y = tanh(x * s) with s [rows, 1]: its grad sums over columns, which the
    run's column sums cannot share a kernel with; the grads are the same."""
    rng = np.random.default_rng(5)
    x = rng.standard_normal((300, 128)).astype(np.float32)
    s = rng.standard_normal((300, 1)).astype(np.float32)
    got = {}
    for jit in (True, False):
        lib.pg_autograd_set_jit(jit)
        try:
            nx, ns = lib.var(x), lib.var(s)
            y = lib.op("tanh", lib.op("mul", nx, ns))
            loss = lib.op("sum_all", y)
            lib.pg_backward(loss)
            got[jit] = (lib.grad(nx), lib.grad(ns), lib.value(loss))
            for n in (loss, y, ns, nx):
                lib.pg_node_free(n)
        finally:
            lib.pg_autograd_set_jit(True)
    for a, b in zip(got[True], got[False]):
        assert np.abs(a - b).max() <= 2e-6 * max(1.0, np.abs(b).max())


def test_grads_accumulate_into_existing_ones(lib):
    """x feeds the run and a product below it, whose grad adds to the one the region wrote."""
    rng = np.random.default_rng(6)
    x = rng.standard_normal((260, 68)).astype(np.float32)
    got = {}
    for jit in (True, False):
        lib.pg_autograd_set_jit(jit)
        try:
            nx = lib.var(x)
            w = lib.var((0.1 * rng.standard_normal((68, 68))).astype(np.float32) if jit else wv)
            wv = lib.value(w)
            y = lib.op("mul", lib.op("matmul", nx, w), nx)
            z = lib.op("tanh", y)
            loss = lib.op("sum_all", z)
            lib.pg_backward(loss)
            got[jit] = (lib.grad(nx), lib.grad(w), lib.value(loss))
            for n in (loss, z, y, w, nx):
                lib.pg_node_free(n)
        finally:
            lib.pg_autograd_set_jit(True)
    for a, b in zip(got[True], got[False]):
        assert np.abs(a - b).max() <= 5e-6 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("cols", [68, 1037, 128])
def test_region_adds_to_an_existing_grad(lib, cols):
    """loss = sum(tanh(x + b) @ w1 + x @ w2): the walk reaches x @ w2 first, so the
    region of tanh and + adds to x's grad (beta 1) beside the bias grad it sums.
    Columns: whole 16-byte pieces that end inside a 128-byte line, odd, and whole
    lines."""
    rng = np.random.default_rng(cols)
    rows, n = 300, 24
    x = rng.standard_normal((rows, cols)).astype(np.float32)
    b = (0.1 * rng.standard_normal(cols)).astype(np.float32)
    w1, w2 = ((cols ** -0.5 * rng.standard_normal((cols, n))).astype(np.float32) for _ in range(2))
    nx, nb, n1, n2 = lib.var(x), lib.var(b), lib.var(w1), lib.var(w2)
    made = [lib.op("add", nx, nb)]
    made.append(lib.op("tanh", made[-1]))
    m1 = lib.op("matmul", made[-1], n1)
    m2 = lib.op("matmul", nx, n2)
    y = lib.op("add", m1, m2)
    loss = lib.op("sum_all", y)
    lib.pg_backward(loss)
    assert lib.pg_autograd_last_was_jit(), lib.pg_autograd_last_error().decode()
    x64, b64, w1d, w2d = (v.astype(np.float64) for v in (x, b, w1, w2))
    t = np.tanh(x64 + b64)
    dt = (1 - t * t) * w1d.sum(1)
    ref = {"dx": dt + w2d.sum(1), "db": dt.sum(0), "dw1": np.repeat(t.sum(0)[:, None], n, 1)}
    # products of 24 terms, tanh and its grad to a few units in the last place, then rows + 16 additions for db
    u = 2.0 ** -24
    mag = np.abs(w1d).sum(1) + np.abs(w2d).sum(1)
    assert (np.abs(lib.grad(nx) - ref["dx"]) <= 64 * u * mag).all()
    assert (np.abs(lib.grad(nb) - ref["db"]) <= (rows + 64) * u * rows * np.abs(w1d).sum(1)).all()
    assert (np.abs(lib.grad(n1) - ref["dw1"]) <= (rows + 64) * u * np.abs(t).sum(0)[:, None]).all()
    for v in (loss, y, m2, m1, *reversed(made), n2, n1, nb, nx):
        lib.pg_node_free(v)


@pytest.mark.parametrize("rows,cols", [(1100, 16), (4100, 4), (700, 24), (9000, 2)])
def test_error_of_few_columns_is_no_larger_than_with_four_row_lanes(lib, rows, cols):
    """y = (x + b) g: db is the column sums of g, exact terms.  The error against
    f64 over at least 1024 sums, beside that of four row lanes over bands of 16 rows
    formed here in f32, as for wide outputs.  By halves the many row lanes measure
    0.9 to 1.05 of it, in one chain 1.5 to 2.2; the ratio of two such norms is good
    to about 4 %."""
    rng = np.random.default_rng(rows)
    e = eo = 0.0
    for _ in range(-(-1024 // cols) if cols > 2 else 300):
        x, g = (rng.standard_normal((rows, cols)).astype(np.float32) for _ in range(2))
        nx, nb, ng = lib.var(x), lib.var(np.zeros(cols, np.float32)), lib.var(g)
        t = lib.op("add", nx, nb)
        y = lib.op("mul", t, ng)
        loss = lib.op("sum_all", y)
        lib.pg_backward(loss)
        got = lib.grad(nb)
        for n in (loss, y, t, ng, nb, nx):
            lib.pg_node_free(n)
        ref = g.astype(np.float64).sum(0)
        pad = np.zeros((-(-rows // 16) * 16, cols), np.float32)
        pad[:rows] = g
        band = pad.reshape(-1, 4, 4, cols)  # 16 rows: lane q takes rows q, q + 4, ...
        lane = ((band[:, 0] + band[:, 1]) + band[:, 2]) + band[:, 3]
        part = ((lane[:, 0] + lane[:, 1]) + lane[:, 2]) + lane[:, 3]
        red = np.zeros((128, cols), np.float32)
        for k in range(0, len(part), 128):
            red[:len(part[k:k + 128])] += part[k:k + 128]
        while len(red) > 1:
            red = red[:len(red) // 2] + red[len(red) // 2:]
        e += float(((got - ref) ** 2).sum())
        eo += float(((red[0] - ref) ** 2).sum())
    assert e <= 1.2 ** 2 * eo, (e / eo) ** 0.5
