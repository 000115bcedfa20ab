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
    """x feeds the run and a second branch: the region adds to x's grad (beta 1)."""
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
