"""Performance cases of the strict owned-tensor path on one GPU.

A case is one call that a program makes with its tensors resident on the GPU: a single
MatMul, a layer, a training step, a parameter update or a loss. Sizes are those of the
repository's configurations and benchmark (the single-layer step, the binary64 layer, the
three-layer MLPs, the 2^28-element update, the published small calls) or generic layer
sizes, whole and ragged. Inputs live in torch tensors that the program lends to the
framework; results come back as torch tensors over the framework's own buffers.
"""
from __future__ import annotations

import functools
import importlib.util
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    if "fusion_pcu_amd" not in sys.modules:
        # The package's folder name has a hyphen, so it is loaded by its path.
        folder = os.path.join(_ROOT, "fusion-pcu_amd")
        spec = importlib.util.spec_from_file_location(
            "fusion_pcu_amd", os.path.join(folder, "__init__.py"), submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["fusion_pcu_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["fusion_pcu_amd"]


pcu = _package()
from fusion_pcu_amd import graph as g  # noqa: E402

_TORCH = {"f32": torch.float32, "f64": torch.float64}
_NUMPY = {"f32": np.dtype(np.float32), "f64": np.dtype(np.float64)}
_SIZE = {"f32": 4, "f64": 8}
_POLICY = {"ieee": 0, "reject_subnormal": 1, "allow_gradual": 2}
_LR = {"layer_step": 0.01, "mlp_step": 1e-3, "sgd": 0.01}


# ------------------------------------------------------------------------- cases


def _matmul(m, k, n, dtype="f32", tl=False, tr=False, policy="ieee", native=False):
    return {"kind": "matmul", "m": m, "k": k, "n": n, "dtype": dtype, "tl": tl, "tr": tr,
            "policy": policy, "native": native}


def _layer(m, k, n, dtype="f32"):
    return {"kind": "layer", "m": m, "k": k, "n": n, "dtype": dtype}


def _layer_step(batch, inputs, outputs, dtype="f32"):
    return {"kind": "layer_step", "batch": batch, "d0": inputs, "d1": outputs, "dtype": dtype}


def _mlp_step(batch, d0, d1, d2, d3, dtype="f32", native=False):
    return {"kind": "mlp_step", "batch": batch, "d0": d0, "d1": d1, "d2": d2, "d3": d3,
            "dtype": dtype, "native": native}


def _elementwise(op, n, dtype="f32"):
    return {"kind": "elementwise", "op": op, "n": n, "dtype": dtype}


def _mse(rows, cols, dtype="f32"):
    return {"kind": "mse", "rows": rows, "cols": cols, "dtype": dtype}


def listed():
    return [
        # The smallest calls: one resident MatMul at a published size, and the single-layer
        # training step (forward, loss, reverse mode, two updates), where latency and
        # launches count.
        dict(_matmul(64, 256, 64), name="matmul_f32_64x256x64"),
        dict(_layer_step(64, 128, 64), name="layer_step_f32_64x128x64"),
        # Inference with a batch of 64 through a wide layer: few output cells, a long sum.
        dict(_matmul(64, 4096, 1024), name="matmul_f32_64x4096x1024"),
        # A weight gradient (op(A) transposed) of ragged layer sizes with subnormal results
        # rejected.
        dict(_matmul(777, 3000, 555, tl=True, policy="reject_subnormal"),
             name="matmul_f32_tn_reject_777x3000x555"),
        # A binary64 input gradient (op(B) transposed) of a middle-sized layer.
        dict(_matmul(1000, 1000, 1000, "f64", tr=True), name="matmul_f64_nt_1000"),
        # The headline MatMul.
        dict(_matmul(4096, 4096, 4096), name="matmul_f32_4096"),
        # A full-size binary64 layer: MatMul, checked bias add, ReLU in one program.
        dict(_layer(4096, 4096, 4096, "f64"), name="layer_f64_4096"),
        # Training steps of three-layer MLPs: a middle-sized one with a batch that is no
        # multiple of a tile, the same sizes with explicitly permitted native compounds, and
        # the full-size loop's step.
        dict(_mlp_step(1000, 1024, 2048, 2048, 1024), name="mlp_step_f32_1000"),
        dict(_mlp_step(1024, 1024, 2048, 2048, 1024, native=True), name="mlp_step_native_f32_1024"),
        dict(_mlp_step(4096, 1024, 4096, 4096, 1024), name="mlp_step_f32_4096"),
        # A parameter update over 2^28 weights, bound by memory.
        dict(_elementwise("sgd", 1 << 28), name="sgd_f32_2p28"),
        # The full-size MLP's loss on its own.
        dict(_mse(4096, 1024), name="mse_f32_4096x1024"),
    ]


def _log_int(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; half of the larger ones whole multiples
    of 64, the rest as they come (odd ones among them)."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    if v >= 128 and rng.random() < 0.5:
        v = (v + 32) // 64 * 64
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choices(("matmul", "layer", "layer_step", "mlp_step", "elementwise", "mse"),
                       weights=(9, 2, 2, 3, 3, 2))[0]
    dtype = "f64" if rng.random() < 0.3 else "f32"
    if kind == "matmul":
        return _matmul(_log_int(rng, 1, 4096), _log_int(rng, 8, 4096), _log_int(rng, 8, 4096),
                       dtype, rng.random() < 0.35, rng.random() < 0.35,
                       rng.choices(("ieee", "reject_subnormal", "allow_gradual"), weights=(8, 2, 1))[0],
                       rng.random() < 0.15)
    if kind == "layer":
        return _layer(_log_int(rng, 16, 4096), _log_int(rng, 16, 4096), _log_int(rng, 16, 4096), dtype)
    if kind == "layer_step":
        return _layer_step(_log_int(rng, 8, 1024), _log_int(rng, 16, 1024), _log_int(rng, 8, 1024), dtype)
    if kind == "mlp_step":
        top = 2048 if dtype == "f32" else 1024
        return _mlp_step(_log_int(rng, 16, 2 * top), *(_log_int(rng, 32, top) for _ in range(4)),
                         dtype, rng.random() < 0.2)
    if kind == "elementwise":
        n = _log_int(rng, 1 << 10, 1 << 28)
        return _elementwise(rng.choice(("sgd", "add", "relu", "relu_backward", "add_relu")),
                            n if dtype == "f32" else max(1 << 10, n // 2), dtype)
    return _mse(_log_int(rng, 16, 4096), _log_int(rng, 8, 4096), dtype)


# ------------------------------------------------------------------------- inputs


class _Inputs:
    """Seeded inputs on the GPU with the configurations' distributions."""

    def __init__(self, case, seed):
        self.dtype = _TORCH[case["dtype"]]
        self.gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)

    def uniform(self, *shape, scale=1.0):
        t = torch.rand(shape, dtype=self.dtype, device="cuda", generator=self.gen)
        return t.mul_(2.0 * scale).sub_(scale)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, dtype=self.dtype, device="cuda", generator=self.gen).mul_(std)

    def xavier(self, fan_in, fan_out):
        return self.uniform(fan_in, fan_out, scale=(6.0 / (fan_in + fan_out)) ** 0.5)


def _tensors(case, seed):
    r, kind = _Inputs(case, seed), case["kind"]
    if kind in ("matmul", "layer"):
        m, k, n = case["m"], case["k"], case["n"]
        make = r.uniform if case["dtype"] == "f32" else r.normal
        if kind == "layer":
            return [make(m, k), make(k, n), make(m, n)]
        return [make(k, m) if case["tl"] else make(m, k), make(n, k) if case["tr"] else make(k, n)]
    if kind == "layer_step":
        b, d0, d1 = case["batch"], case["d0"], case["d1"]
        return [r.uniform(b, d0), r.uniform(d0, d1), r.uniform(b, d1), r.uniform(b, d1)]
    if kind == "mlp_step":
        d = [case["d%d" % i] for i in range(4)]
        return [r.uniform(case["batch"], d[0]), r.xavier(d[0], d[1]), r.xavier(d[1], d[2]),
                r.xavier(d[2], d[3]), r.uniform(case["batch"], d[3])]
    if kind == "elementwise":
        n, op = case["n"], case["op"]
        if op == "sgd":
            return [r.normal(n), r.normal(n, std=1e-3)]
        return [r.normal(n)] if op == "relu" else [r.normal(n), r.normal(n)]
    # A prediction before the first update against its target.
    return [r.normal(case["rows"], case["cols"], std=0.3), r.uniform(case["rows"], case["cols"])]


# ------------------------------------------------------------ the program's handles


@functools.lru_cache(maxsize=None)
def _function(kind, native):
    """The program's captured functions: each is defined once and called on every state."""
    if kind == "layer_step":
        return g.c1_training_step(_LR[kind])
    if kind == "mlp_step":
        return g.mlp_training_step(_LR[kind], native=native)

    @g.function(strict=True)
    def layer(x, w, b):
        return g.relu(g.add(g.matmul(x, w), b))

    return layer


def _array(t):
    """A torch tensor lent to the framework."""
    return pcu.DeviceArray(g.default_context(), t.data_ptr(), tuple(t.shape),
                           _NUMPY["f32" if t.dtype == torch.float32 else "f64"])


class _Held:
    """A framework-owned result seen by torch without a copy; the tensor keeps it alive."""

    def __init__(self, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {
            "shape": owner.shape, "typestr": owner.dtype.str, "data": (owner.array.ptr, False),
            "strides": None, "version": 2}


def _tensor(owner):
    return torch.as_tensor(_Held(owner), device="cuda")


def prepare(case, seed):
    tensors = _tensors(case, seed)
    kind = case["kind"]
    state = {"case": case, "keep": tensors}
    if kind in ("layer", "layer_step", "mlp_step"):
        state["function"] = _function(kind, bool(case.get("native")))
        state["args"] = [g.PcuTensor(_array(t), owned=False) for t in tensors]
    else:
        dtype = tensors[0].dtype
        shape = {"matmul": lambda: (case["m"], case["n"]), "mse": lambda: (),
                 "elementwise": lambda: (case["n"],)}[kind]()
        state["result"] = torch.empty(shape, dtype=dtype, device="cuda")
        state["args"] = [_array(t) for t in tensors]
        state["out"] = _array(state["result"])
    torch.cuda.synchronize()  # the inputs exist before the framework's own stream reads them
    return state


def run(state):
    case, args = state["case"], state["args"]
    kind = case["kind"]
    if kind == "layer":
        return _tensor(state["function"](*args))
    if kind in ("layer_step", "mlp_step"):
        return [_tensor(t) for t in state["function"](*args)]
    ctx, out = g.default_context(), state["out"]
    if kind == "matmul":
        if case["native"]:
            ctx.native_matmul(args[0], args[1], case["tl"], case["tr"], out=out)
        else:
            ctx.strict_matmul(args[0], args[1], case["tl"], case["tr"], _POLICY[case["policy"]], out=out)
    elif kind == "mse":
        ctx.strict_mse(args[0], args[1], out=out)
    elif case["op"] == "sgd":
        ctx.strict_sgd(args[0], args[1], _LR["sgd"], out=out)
    elif case["op"] == "add":
        ctx.checked_binary(0, args[0], args[1], out=out)
    elif case["op"] == "relu":
        ctx.checked_relu(args[0], out=out)
    elif case["op"] == "relu_backward":
        ctx.checked_relu_backward(args[0], args[1], out=out)
    else:
        ctx.checked_add_relu(args[0], args[1], out=out)
    return state["result"]


# ------------------------------------------------------------- work and tolerances


def work(case):
    kind, size = case["kind"], _SIZE[case["dtype"]]
    if kind in ("matmul", "layer"):
        m, k, n = case["m"], case["k"], case["n"]
        extra = m * n if kind == "layer" else 0
        return {"bytes": size * (m * k + k * n + m * n + extra), "flops": 2 * m * n * k + 2 * extra}
    if kind == "layer_step":
        b, d0, d1 = case["batch"], case["d0"], case["d1"]
        return {"bytes": size * (b * d0 + 2 * d0 * d1 + 3 * b * d1 + 1),
                "flops": 4 * b * d0 * d1 + 2 * d0 * d1 + 11 * b * d1}
    if kind == "mlp_step":
        b, d = case["batch"], [case["d%d" % i] for i in range(4)]
        pairs = [d[0] * d[1], d[1] * d[2], d[2] * d[3]]
        return {"bytes": size * (b * (d[0] + d[3]) + 2 * sum(pairs) + 1),
                "flops": 2 * b * (2 * sum(pairs) + pairs[1] + pairs[2]) + 2 * sum(pairs) + 5 * b * d[3]}
    if kind == "elementwise":
        n, op = case["n"], case["op"]
        return {"bytes": size * n * (2 if op == "relu" else 3),
                "flops": n * {"sgd": 2, "add": 1, "relu": 1, "relu_backward": 1, "add_relu": 2}[op]}
    n = case["rows"] * case["cols"]
    return {"bytes": size * (2 * n + 1), "flops": 3 * n}


def tolerance(case):
    """Every strict operation has one result: order and rounding are fixed by the contract.
    A native compound leaves both to the backend."""
    if not case.get("native"):
        return "exact"
    # About four times the distance from binary64 (sums of a few thousand terms: 1e-6 and 2e-15;
    # an updated weight: half an ulp, the change of its gradient's sums vanishing beside it).
    f32 = case["dtype"] == "f32"
    if case["kind"] == "mlp_step":
        return {"rel": 4e-7, "max": 1e-5} if f32 else {"rel": 8e-15, "max": 1e-13}
    return {"rel": 5e-6, "max": 5e-5} if f32 else {"rel": 1e-14, "max": 1e-13}


def exact(case, seed):
    """The same call in binary64 by plain torch."""
    t = [x.double() for x in _tensors(case, seed)]
    kind = case["kind"]
    if kind == "matmul":
        a, b = (t[0].t() if case["tl"] else t[0]), (t[1].t() if case["tr"] else t[1])
        return a.contiguous() @ b.contiguous()
    if kind == "layer":
        return torch.relu(t[0] @ t[1] + t[2])
    if kind == "mse":
        return ((t[0] - t[1]) ** 2).mean()
    if kind == "elementwise":
        op = case["op"]
        if op == "sgd":
            return t[0] - float(np.float32(_LR["sgd"])) * t[1]
        if op == "relu":
            return torch.relu(t[0])
        if op == "relu_backward":
            return torch.where(t[0] > 0, t[1], torch.zeros_like(t[1]))
        return t[0] + t[1] if op == "add" else torch.relu(t[0] + t[1])
    lr = float(np.float32(_LR[kind]))
    if kind == "layer_step":
        x, w, b, y = t
        z = x @ w + b
        h = torch.relu(z)
        d = torch.where(z > 0, (h - y) * (2.0 / y.numel()), torch.zeros_like(z))
        return [w - lr * (x.t().contiguous() @ d), b - lr * d, ((h - y) ** 2).mean()]
    x, w1, w2, w3, y = t
    m1 = x @ w1
    h1 = torch.relu(m1)
    m2 = h1 @ w2
    h2 = torch.relu(m2)
    p = h2 @ w3
    d3 = (p - y) * (2.0 / y.numel())
    d2 = torch.where(m2 > 0, d3 @ w3.t().contiguous(), torch.zeros_like(m2))
    d1 = torch.where(m1 > 0, d2 @ w2.t().contiguous(), torch.zeros_like(m1))
    return [w1 - lr * (x.t().contiguous() @ d1), w2 - lr * (h1.t().contiguous() @ d2),
            w3 - lr * (h2.t().contiguous() @ d3), ((p - y) ** 2).mean()]
