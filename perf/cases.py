"""The work that programs built on this library give it, as cases to time.

Every case goes through the C ABI the way a program does (autograd nodes,
pg_backward, the optimisers), on tensors that already live in HBM.  A case is
a dict of plain values with a "kind":

  chain     tanh(relu((a + b) * c)) over small leaves made from host arrays,
            sum_all, pg_backward: the smallest call, launch-bound
  gate      gelu(x + bias) * sigmoid(g) over resident tensors, sum_all,
            pg_backward: a broadcasting elementwise graph, memory-bound
  matmul    pg_ag_matmul in f32, f16 or bf16, plain or batched, forward and
            both grads of a given upstream grad
  linear    pg_amd_ag_linear16: one mixed-precision layer, forward and the
            grads of x, W and b
  mlp_step  a whole training step of an MLP with gelu layers: zero_grad,
            forward, mse, pg_backward, pg_sgd_step
  mlp_infer the same network's forward without grads
  optim     new grads, pg_clip_grad_norm and one optimiser step over an
            MLP's parameters

prepare() makes what a program holds before the call (leaves, weights, an
optimiser), run() makes one pass and returns views of the device tensors it
leaves, exact() gives the same values in 64-bit arithmetic.  The 16-bit layers
define their result on operands rounded to 16 bits (nearest even), so exact()
rounds the same operands and computes everything else in 64 bits.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import picograd_amd
from picograd_amd.capi import BF16, F16, F32, AdamCfg, PgNode, PgTensorAmd, SgdCfg, shape_arg
from picograd_amd.mlp import ACT_GELU, ACT_NONE, ACT_RELU, Mlp

DTYPES = {"f32": F32, "f16": F16, "bf16": BF16}
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16}
ACTS = {"none": ACT_NONE, "relu": ACT_RELU, "gelu": ACT_GELU}
CLIP_SHARE = 0.9  # max_norm of the optim cases over the grads' norm, so that every step scales
SGD = {"momentum": 0.9, "weight_decay": 1e-4}
ADAM = {"lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8, "weight_decay": 0.01}

# the largest products that draw() asks for, in multiply-adds
MOST = {"f32": 1 << 31, "f16": 8192 * 4096 * 4096, "bf16": 8192 * 4096 * 4096}
MOST_PARAMS = 37_801_994  # those of the largest network


def listed() -> list[dict]:
    return [
        # the loop of the reference's JIT benchmark: leaves from host arrays, forward, sum, backward
        {"name": "chain-64x64", "kind": "chain", "rows": 64, "cols": 64},
        # the fused broadcasting backward that the benchmark's headline is quoted on, with its forward
        {"name": "gate-16384x4096", "kind": "gate", "rows": 16384, "cols": 4096},
        # the same graph at an ordinary size that no vector width divides
        {"name": "gate-3001x1037", "kind": "gate", "rows": 3001, "cols": 1037},
        # a large bf16 product with both grads
        {"name": "matmul-bf16-8192x4096x4096", "kind": "matmul", "dtype": "bf16", "batch": 1,
         "m": 8192, "k": 4096, "n": 4096},
        # ragged f16: no dimension fits a tile
        {"name": "matmul-f16-4097x1000x3000", "kind": "matmul", "dtype": "f16", "batch": 1,
         "m": 4097, "k": 1000, "n": 3000},
        # attention-style scores: many small products
        {"name": "bmm-f16-32x512x128x512", "kind": "matmul", "dtype": "f16", "batch": 32,
         "m": 512, "k": 128, "n": 512},
        # the reference's own dtype, which a program has before it asks for another
        {"name": "matmul-f32-2048x1024x1024", "kind": "matmul", "dtype": "f32", "batch": 1,
         "m": 2048, "k": 1024, "n": 1024},
        # one hidden layer at an ordinary batch
        {"name": "linear-bf16-512x1024x4096", "kind": "linear", "dtype": "bf16", "act": "gelu",
         "m": 512, "k": 1024, "n": 4096},
        # a small f32 network on flattened images, as picograd's own examples train theirs
        {"name": "mlp-step-f32-784x512x256x10", "kind": "mlp_step", "dtype": "f32", "fused": False, "batch": 256,
         "dims": "784x512x256x10"},
        # the benchmark's training step
        {"name": "mlp-step-bf16-b4096", "kind": "mlp_step", "dtype": "bf16", "fused": True, "batch": 4096,
         "dims": "1024x4096x4096x4096x10"},
        # serving the same network: a few rows against all of its weights
        {"name": "mlp-infer-bf16-b16", "kind": "mlp_infer", "dtype": "bf16", "batch": 16,
         "dims": "1024x4096x4096x4096x10"},
        # clipping and AdamW over that network's parameters
        {"name": "adamw-clip-37.8M", "kind": "optim", "opt": "adamw", "dims": "1024x4096x4096x4096x10"},
    ]


def _log(rng, lo: int, hi: int) -> int:
    """Whole number from lo to hi, even over its logarithm; 8's multiples half of the time where they fit."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 16 and rng.random() < 0.5:
        v -= v % 8
    return min(max(v, lo), hi)


def _dims(rng, lo: int, hi: int) -> list[int]:
    return [_log(rng, lo, hi) for _ in range(rng.randint(2, 4))] + [_log(rng, 1, 64)]


def _weights(dims) -> int:
    return sum(a * b for a, b in zip(dims, dims[1:]))


def draw(rng) -> dict:
    kind = rng.choice(["chain", "gate", "matmul", "matmul", "linear", "mlp_step", "mlp_infer", "optim"])
    while True:
        if kind == "chain":
            return {"kind": kind, "rows": _log(rng, 1, 256), "cols": _log(rng, 1, 256)}
        if kind == "gate":
            c = {"kind": kind, "rows": _log(rng, 16, 16384), "cols": _log(rng, 16, 8192)}
            if c["rows"] * c["cols"] <= 1 << 26:
                return c
        elif kind == "matmul":
            c = {"kind": kind, "dtype": rng.choice(["f32", "f16", "bf16"]),
                 "batch": 1 if rng.random() < 0.7 else _log(rng, 2, 64),
                 "m": _log(rng, 8, 8192), "k": _log(rng, 8, 4096), "n": _log(rng, 8, 4096)}
            if c["batch"] * c["m"] * c["k"] * c["n"] <= MOST[c["dtype"]] and c["batch"] * c["m"] <= 1 << 16:
                return c
        elif kind == "linear":
            c = {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "act": rng.choice(["none", "relu", "gelu"]),
                 "m": _log(rng, 8, 4096), "k": _log(rng, 8, 4096), "n": _log(rng, 8, 4096)}
            return c
        elif kind == "mlp_step":
            dt = rng.choice(["f32", "f16", "bf16"])
            batch, dims = _log(rng, 16, 4096), _dims(rng, 16, 4096)
            if batch * _weights(dims) <= (1 << 31 if dt == "f32" else 1 << 37):
                return {"kind": kind, "dtype": dt, "fused": dt != "f32" and rng.random() < 0.7, "batch": batch,
                        "dims": "x".join(map(str, dims))}
        elif kind == "mlp_infer":
            return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "batch": _log(rng, 1, 1024),
                    "dims": "x".join(map(str, _dims(rng, 64, 4096)))}
        else:
            dims = _dims(rng, 64, 4096)
            if _weights(dims) <= MOST_PARAMS:
                return {"kind": kind, "opt": rng.choice(["sgd", "adam", "adamw", "amsgrad"]),
                        "dims": "x".join(map(str, dims))}


# ---------------------------------------------------------------- inputs
# made from the seed alone, in the order below, so that prepare() and exact()
# have the same ones

def _gen(seed: int, device="cuda") -> torch.Generator:
    return torch.Generator(device=device).manual_seed(int(seed))


def _normal(g, shape, std=1.0) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=g.device) * std


def _uniform(g, shape, lim) -> torch.Tensor:
    return (torch.rand(shape, generator=g, device=g.device) * 2 - 1) * lim


def _dims_of(case) -> list[int]:
    return [int(d) for d in case["dims"].split("x")]


def _inputs(case, seed) -> dict:
    kind = case["kind"]
    if kind == "chain":  # host arrays
        g = _gen(seed, "cpu")
        return {k: _uniform(g, (case["rows"], case["cols"]), 1.0) for k in "abc"}
    g = _gen(seed)
    if kind == "gate":
        n = (case["rows"], case["cols"])
        return {"x": _normal(g, n), "bias": _normal(g, n[1:], 0.1), "g": _normal(g, n)}
    if kind == "matmul":
        b = () if case["batch"] == 1 else (case["batch"],)
        m, k, n = case["m"], case["k"], case["n"]
        # a batched product is one of scores, whose operands have 1/sqrt(k) variance; a plain one is a weight's
        sa, sb = (k ** -0.5, k ** -0.5) if b else (1.0, 0.02)
        v = {"a": _normal(g, b + (m, k), sa), "b": _normal(g, b + (k, n), sb)}
        if case["dtype"] != "f32":
            v = {q: t.to(TORCH[case["dtype"]]) for q, t in v.items()}
        v["dc"] = _normal(g, b + (m, n))
        return v
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": _normal(g, (m, k)), "w": _uniform(g, (k, n), k ** -0.5), "b": _normal(g, (n,), 0.1),
                "dout": _normal(g, (m, n))}
    d = _dims_of(case)
    v = {}
    for i, (a, b) in enumerate(zip(d, d[1:])):
        v["w%d" % i] = _uniform(g, (a, b), a ** -0.5)
        v["b%d" % i] = _uniform(g, (b,), a ** -0.5)
    if kind == "optim":
        v.update({"g" + q: _normal(g, t.shape, 0.05) for q, t in list(v.items())})
        return v
    v["x"] = _normal(g, (case["batch"], d[0]))
    if kind == "mlp_step":
        v["target"] = _normal(g, (case["batch"], d[-1]))
    return v


# ---------------------------------------------------------------- state

_GRAD_AT, _DEV_AT = PgNode.grad.offset, PgTensorAmd.dev.offset


class _Memory:
    """Device memory of the library, for torch."""

    def __init__(self, ptr: int, shape, kind: str):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": kind, "version": 3,
                                         "strides": None}


def _view(ptr: int, shape, kind="<f4") -> torch.Tensor:
    return torch.as_tensor(_Memory(ptr, shape, kind), device="cuda")


class _State:
    """What one program holds: long-lived nodes and tensors, and the nodes of
    its latest pass, which go when the next one begins."""

    def __init__(self, lib, case):
        self.L, self.case = lib, case
        self.nodes, self.tensors, self.frees, self.last, self.views = [], [], [], [], {}

    def tensor(self, t: torch.Tensor) -> int:
        """Device tensor with t's elements."""
        nd, sh = shape_arg(t.shape)
        code = {torch.float32: F32, torch.float16: F16, torch.bfloat16: BF16}[t.dtype]
        p = self.L.pg_tensor_empty_dtype(code, nd, sh)
        if not p:
            raise RuntimeError(self.L.pg_amd_last_error().decode())
        self.L.sync()
        if t.dtype == torch.float32:
            _view(self.dev(p), t.shape).copy_(t)
        else:
            _view(self.dev(p), t.shape, "<i2").copy_(t.view(torch.int16))
        torch.cuda.synchronize()
        self.L.pg_amd_tensor_modified(p)
        return p

    def var(self, t: torch.Tensor, requires_grad=True) -> int:
        p = self.tensor(t)
        n = self.L._check(self.L.pg_var_from_tensor(p, requires_grad))
        self.L.pg_tensor_free(p)
        self.nodes.append(n)
        return n

    @staticmethod
    def dev(tensor: int) -> int:
        return C.c_void_p.from_address(tensor + _DEV_AT).value

    def out(self, tensor: int, shape) -> torch.Tensor:
        ptr = self.dev(tensor)
        got = self.views.get((ptr, shape))
        if got is None:
            if len(self.views) > 256:
                self.views.clear()
            got = self.views[ptr, shape] = _view(ptr, shape)
        return got

    def value(self, node: int, shape) -> torch.Tensor:
        return self.out(C.c_void_p.from_address(node).value, shape)

    def grad(self, node: int, shape) -> torch.Tensor:
        return self.out(C.c_void_p.from_address(node + _GRAD_AT).value, shape)

    def drop(self) -> None:
        for n in reversed(self.last):
            self.L.pg_node_free(n)
        self.last = []

    def __del__(self):
        self.drop()
        self.views = {}
        for f, p in self.frees:
            f(p)
        for t in self.tensors:
            self.L.pg_tensor_free(t)
        for n in self.nodes:
            self.L.pg_node_free(n)


_LIB = []


def _lib():
    if not _LIB:
        L = picograd_amd.load()
        if L.pg_amd_init() != 0:
            raise RuntimeError(L.pg_amd_last_error().decode())
        _LIB.append(L)
    return _LIB[0]


def prepare(case, seed) -> _State:
    L = _lib()
    s = _State(L, case)
    v = _inputs(case, seed)
    kind = case["kind"]
    if kind == "chain":
        s.host = [np.ascontiguousarray(v[k].numpy(), np.float32) for k in "abc"]
        s.ptrs = [h.ctypes.data for h in s.host]
        s.ndim, s.shape_c = shape_arg((case["rows"], case["cols"]))
    elif kind == "gate":
        s.x, s.bias, s.g = (s.var(v[k]) for k in ("x", "bias", "g"))
    elif kind == "matmul":
        s.a, s.b = s.var(v["a"]), s.var(v["b"])
        s.dc = s.tensor(v["dc"])
        s.tensors.append(s.dc)
    elif kind == "linear":
        s.x, s.w, s.b = (s.var(v[k]) for k in ("x", "w", "b"))
        s.dout = s.tensor(v["dout"])
        s.tensors.append(s.dout)
    else:
        d = _dims_of(case)
        s.dims, s.layers = d, len(d) - 1
        s.ws = [s.var(v["w%d" % i]) for i in range(s.layers)]
        s.bs = [s.var(v["b%d" % i]) for i in range(s.layers)]
        s.shapes = {"w%d" % i: (d[i], d[i + 1]) for i in range(s.layers)}
        s.shapes.update({"b%d" % i: (d[i + 1],) for i in range(s.layers)})
        s.params = {"w%d" % i: w for i, w in enumerate(s.ws)}
        s.params.update({"b%d" % i: b for i, b in enumerate(s.bs)})
        if kind == "optim":
            _prepare_optim(s, v)
        else:
            s.x = s.var(v["x"], False)
            s.xv = C.c_void_p.from_address(s.x).value
            # mse's mean is over the last axis alone, so the loss and its grads grow with the batch
            lr = 0.01 / case["batch"]
            for n in s.ws + s.bs:
                L.pg_node_retain(n)  # the network frees its parameters itself
            s.mlp = Mlp(L, s.ws, s.bs, DTYPES[case["dtype"]], sgd=(lr, SGD["momentum"], 0.0, SGD["weight_decay"], True),
                        fused=bool(case.get("fused", case["dtype"] != "f32")))
            s.frees.append((lambda m: m.free(), s.mlp))
            if kind == "mlp_step":
                s.target = s.var(v["target"], False)
    L.sync()
    torch.cuda.synchronize()
    return s


def _prepare_optim(s, v) -> None:
    L, case = s.L, s.case
    s.fresh, s.grads, norm2 = [], [], 0.0
    for q, n in s.params.items():
        fresh = s.tensor(v["g" + q])
        s.tensors.append(fresh)
        s.fresh.append(fresh)
        L.node(n).grad = L.pg_tensor_clone(fresh)  # the node owns it
        s.grads.append(L.node(n).grad)
        norm2 += float(v["g" + q].double().square().sum())
    s.max_norm = CLIP_SHARE * math.sqrt(norm2)
    s.arr = (C.c_void_p * len(s.params))(*s.params.values())
    if case["opt"] == "sgd":
        s.opt = L.pg_sgd_new(C.byref(SgdCfg(0.01, SGD["momentum"], 0.0, SGD["weight_decay"], True)))
        add, s.step, free = L.pg_sgd_add_param, L.pg_sgd_step, L.pg_sgd_free
    else:
        s.opt = L.pg_adam_new(C.byref(AdamCfg(ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"],
                                              ADAM["weight_decay"], case["opt"] == "amsgrad", case["opt"] != "adam")))
        add, s.step, free = L.pg_adam_add_param, L.pg_adam_step, L.pg_adam_free
    s.frees.append((free, s.opt))
    for n in s.params.values():
        if add(s.opt, n) != 0:
            raise RuntimeError("optimiser: add_param failed")


# ---------------------------------------------------------------- one pass

def run(s) -> dict:
    s.drop()
    out = _RUN[s.case["kind"]](s)
    s.L.pg_amd_stream()  # the results go to whatever the program queues next: nothing stays deferred
    return out


def _run_chain(s):
    L, nd, sh, shape = s.L, s.ndim, s.shape_c, (s.case["rows"], s.case["cols"])
    a, b, c = (L.pg_var_from_data(nd, sh, p, True) for p in s.ptrs)
    t0 = L.pg_ag_add(a, b)
    t1 = L.pg_ag_mul(t0, c)
    t2 = L.pg_ag_relu(t1)
    y = L.pg_ag_tanh(t2)
    loss = L._check(L.pg_ag_sum_all(y))
    L.pg_backward(loss)
    s.last = [a, b, c, t0, t1, t2, y, loss]
    return {"y": s.value(y, shape), "loss": s.value(loss, (1,)), "da": s.grad(a, shape), "db": s.grad(b, shape),
            "dc": s.grad(c, shape)}


def _run_gate(s):
    L, shape = s.L, (s.case["rows"], s.case["cols"])
    t0 = L.pg_ag_add(s.x, s.bias)
    t1 = L.pg_ag_gelu(t0)
    t2 = L.pg_ag_sigmoid(s.g)
    y = L.pg_ag_mul(t1, t2)
    loss = L._check(L.pg_ag_sum_all(y))
    L.pg_backward(loss)
    s.last = [t0, t1, t2, y, loss]
    return {"y": s.value(y, shape), "loss": s.value(loss, (1,)), "dx": s.grad(s.x, shape), "dg": s.grad(s.g, shape),
            "dbias": s.grad(s.bias, shape[1:])}


def _run_matmul(s):
    c = s.case
    b, m, k, n = () if c["batch"] == 1 else (c["batch"],), c["m"], c["k"], c["n"]
    y = s.L._check(s.L.pg_ag_matmul(s.a, s.b))
    s.L.pg_amd_backward_from(y, s.dc)
    s.last = [y]
    return {"c": s.value(y, b + (m, n)), "da": s.grad(s.a, b + (m, k)), "db": s.grad(s.b, b + (k, n))}


def _run_linear(s):
    L, c = s.L, s.case
    m, k, n, act = c["m"], c["k"], c["n"], ACTS[c["act"]]
    L.pg_amd_tensor_modified(C.c_void_p.from_address(s.x).value)  # another batch in the same tensor
    y = L._check(L.pg_amd_ag_linear16(s.x, s.w, s.b, act, DTYPES[c["dtype"]]))
    L.pg_amd_backward_from(y, s.dout)
    s.last = [y]
    # a layer with an activation keeps its pre-activation and forms its output when it is read
    z = L.pg_amd_linear16_preact(y) if act else C.c_void_p.from_address(y).value
    return {"z": s.out(z, (m, n)), "dx": s.grad(s.x, (m, k)), "dw": s.grad(s.w, (k, n)), "db": s.grad(s.b, (n,))}


def _run_mlp_step(s):
    L, m = s.L, s.mlp
    L.pg_amd_tensor_modified(s.xv)  # another batch in the same tensor
    L.pg_sgd_zero_grad(m.opt)
    y, made = m.forward(s.x)
    loss = L._check(L.pg_ag_mse(y, s.target, True))
    L.pg_backward(loss)
    L.pg_sgd_step(m.opt)
    for n in reversed(made[:-1]):
        L.pg_node_free(n)
    s.last = [y, loss]
    out = {"y": s.value(y, (s.case["batch"], s.dims[-1])), "loss": s.value(loss, (1,))}
    for q, n in s.params.items():
        out["d" + q] = s.grad(n, s.shapes[q])
        out[q] = s.value(n, s.shapes[q])
    return out


def _run_mlp_infer(s):
    L = s.L
    L.pg_amd_tensor_modified(s.xv)  # another request in the same tensor
    L.pg_no_grad_push()
    y, made = s.mlp.forward(s.x)
    L.pg_no_grad_pop()
    for n in reversed(made[:-1]):
        L.pg_node_free(n)
    s.last = [y]
    return {"y": s.value(y, (s.case["batch"], s.dims[-1]))}


def _run_optim(s):
    L = s.L
    for g, fresh in zip(s.grads, s.fresh):
        L.pg_tensor_copy_from(g, fresh)  # this step's grads
    norm = L.pg_clip_grad_norm(s.arr, len(s.params), s.max_norm, 1e-6)
    s.step(s.opt)
    out = {q: s.value(n, s.shapes[q]) for q, n in s.params.items()}
    out["norm"] = float(norm)
    return out


_RUN = {"chain": _run_chain, "gate": _run_gate, "matmul": _run_matmul, "linear": _run_linear,
        "mlp_step": _run_mlp_step, "mlp_infer": _run_mlp_infer, "optim": _run_optim}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case) -> dict:
    kind = case["kind"]
    if kind == "chain":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * 7 * n, "flops": 20 * n}
    if kind == "gate":  # x, g in; y, dx, dg out
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (5 * n + 2 * case["cols"]), "flops": 60 * n}
    if kind == "matmul":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": b * (e * (m * k + k * n) + 4 * (2 * m * n + m * k + k * n)), "flops": 6 * b * m * k * n}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (2 * m * n + 2 * m * k + k * n + 2 * n) + 2 * k * n, "flops": 6 * m * k * n}
    d = _dims_of(case)
    params = _weights(d) + sum(d[1:])
    if kind == "optim":  # p, this step's grad and the state in; p, the clipped grad and the state out
        return {"bytes": {"sgd": 24, "adam": 32, "adamw": 32, "amsgrad": 40}[case["opt"]] * params,
                "flops": 15 * params}
    b = case["batch"]
    if kind == "mlp_infer":
        return {"bytes": 2 * _weights(d) + 4 * (sum(d[1:]) + b * (d[0] + d[-1])), "flops": 2 * b * _weights(d)}
    # the first layer's input has no grad; p and its momentum in and out, the grad out
    return {"bytes": 20 * params + 4 * b * (d[0] + 2 * d[-1]), "flops": b * (6 * _weights(d) - 2 * d[0] * d[1])}


def tolerance(case):
    kind = case["kind"]
    if kind == "matmul":
        return {"rel": 1e-5, "max": 1e-4}  # sums of up to 65536 f32 terms in another order
    if kind == "linear":
        # dz is rounded to 16 bits: a last-bit difference of the f32 sums moves a few of its values by one unit,
        # and takes a relu that sits on zero to its other side
        return {"rel": 2e-3, "max": 0.3} if case["act"] == "relu" else {"rel": 1e-4, "max": 2e-2}
    if kind in ("mlp_step", "mlp_infer"):
        # 16-bit roundings of every layer's operands, each moved by the sums before it
        if case["dtype"] == "f32":
            return {"rel": 1e-5, "max": 4e-4}
        return {"rel": 2e-3, "max": 0.1} if kind == "mlp_infer" else {"rel": 6e-3, "max": 0.2}
    if kind == "optim":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-6, "max": 2e-5}  # elementwise f32, and its sums in another order


# ---------------------------------------------------------------- the same values in 64 bits

def _gelu(z):
    return 0.5 * z * (1 + torch.erf(z * 0.5 ** 0.5))


def _gelu_grad(z):
    return 0.5 * (1 + torch.erf(z * 0.5 ** 0.5)) + z * torch.exp(-0.5 * z * z) / math.sqrt(2 * math.pi)


def _q(t, dtype):
    """Rounded to the 16-bit type that the products take, or as it is for f32."""
    return t.to(TORCH[dtype]).double() if dtype in TORCH else t


def _t(t):
    return t.transpose(-1, -2).contiguous()


def exact(case, seed):
    kind = case["kind"]
    v = {k: t.double() for k, t in _inputs(case, seed).items()}
    if kind == "chain":
        s, c = v["a"] + v["b"], v["c"]
        y = torch.tanh(torch.relu(s * c))
        d = (1 - y * y) * (s * c > 0)
        return {"y": y, "loss": y.sum().reshape(1), "da": d * c, "db": d * c, "dc": d * s}
    if kind == "gate":
        z, sg = v["x"] + v["bias"], torch.sigmoid(v["g"])
        h = _gelu(z)
        y = h * sg
        dx = _gelu_grad(z) * sg
        return {"y": y, "loss": y.sum().reshape(1), "dx": dx, "dg": h * sg * (1 - sg), "dbias": dx.sum(0)}
    if kind == "matmul":
        dc = _q(v["dc"], case["dtype"])
        return {"c": v["a"] @ v["b"], "da": dc @ _t(v["b"]), "db": _t(v["a"]) @ dc}
    if kind == "linear":
        dt = case["dtype"]
        x, w = _q(v["x"], dt), _q(v["w"], dt)
        z = x @ w + v["b"]
        dz = v["dout"] * (_gelu_grad(z) if case["act"] == "gelu" else (z > 0).double() if case["act"] == "relu" else 1)
        q = _q(dz, dt)
        return {"z": z, "dx": q @ _t(w), "dw": _t(x) @ q, "db": dz.sum(0)}
    if kind == "optim":
        return _exact_optim(case, v)
    return _exact_mlp(case, v)


def _exact_optim(case, v):
    names = [q for q in v if not q.startswith("g")]
    norm = math.sqrt(sum(float(v["g" + q].square().sum()) for q in names))
    out = {}
    for q in names:
        p, g = v[q], v["g" + q] * (CLIP_SHARE * norm / (norm + 1e-6))
        if case["opt"] == "sgd":
            g = g + SGD["weight_decay"] * p
            out[q] = p - 0.01 * (1 + SGD["momentum"]) * g
            continue
        wd, lr = ADAM["weight_decay"], ADAM["lr"]
        if case["opt"] == "adam":
            g = g + wd * p
        else:
            p = p * (1 - lr * wd)
        out[q] = p - lr * g / (g.abs() + ADAM["eps"])  # the first step: both moments are the grad's own
    out["norm"] = torch.tensor(norm, dtype=torch.float64)
    return out


def _exact_mlp(case, v):
    dt, d = case["dtype"], _dims_of(case)
    n = len(d) - 1
    w = [v["w%d" % i] for i in range(n)]
    qw = [_q(t, dt) for t in w]
    h, hs, zs = v["x"], [], []
    for i in range(n):
        hs.append(_q(h, dt))
        zs.append(hs[i] @ qw[i] + v["b%d" % i])
        h = _gelu(zs[i]) if i + 1 < n else zs[i]
    if case["kind"] == "mlp_infer":
        return {"y": h}
    diff = h - v["target"]
    out = {"y": h, "loss": (diff.square().sum() / d[-1]).reshape(1)}
    dh = 2 * diff / d[-1]
    for i in reversed(range(n)):
        dz = dh * _gelu_grad(zs[i]) if i + 1 < n else dh
        q = _q(dz, dt)
        out["db%d" % i], out["dw%d" % i] = dz.sum(0), _t(hs[i]) @ q
        if i:
            dh = q @ _t(qw[i])
    lr = 0.01 / case["batch"]
    for i in range(n):
        for k in ("w%d" % i, "b%d" % i):
            g = out["d" + k] + SGD["weight_decay"] * v[k]
            out[k] = v[k] - lr * (1 + SGD["momentum"]) * g
    return out
