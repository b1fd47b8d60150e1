"""What a program that trains with this backend has it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` gives the fixed ones, ``draw(rng)`` one more of the same ranges,
``prepare`` makes what a program holds before the call, ``run`` is one pass through the public entry points, ``work`` the
bytes and operations that the pass cannot do without, ``exact`` the same results in 64 bits from plain torch, and
``tolerance`` how far two correct implementations may be apart.

Kinds
-----
train     the fixed training plan (``GpuMlp``): ``steps`` steps, each on a fresh resident batch, then the loss and the
          weights are read, as at the end of an epoch.
linear    one Dense layer through the op-level calls: ``forward`` (bias and ReLU in the epilogue), ``backward``
          (dW, db and dX in one call) or ``layer`` (forward, then the masked backward of a hidden layer).
splitk    the weight and bias gradient of a narrow layer over a long batch, cut into K slices.
tape      an epoch of a Sequential model on the autodiff tape, then its loss: minibatches, Adam, softmax cross-entropy.
softmax   row softmax and its VJP, as the tape's softmax node issues them.
adam      one Adam update of a parameter list.
"""
import ctypes
import math

import torch

from rgpu_amd import autograd as A
from rgpu_amd import gpu as G

# ------------------------------------------------------------------ the cases

_LISTED = [
    # The reference's first workload (its published batch-32 step): a small model and batch, a chain of short launches.
    {"name": "train_f32_b32_sgd", "kind": "train", "dims": "512-1024-1024-10", "batch": 32, "optimizer": "sgd",
     "precision": "f32", "lr": 0.01, "steps": 200},
    # The headline: Adam steps of the same model at batch 2048 (few enough that two correct runs stay comparable).
    {"name": "train_f32_b2048_adam", "kind": "train", "dims": "512-1024-1024-10", "batch": 2048, "optimizer": "adam",
     "precision": "f32", "lr": 1e-3, "steps": 32},
    # Mixed precision with a 1000-class output layer, whose width is no multiple of a tile.
    {"name": "train_bf16_b4096_adam", "kind": "train", "dims": "1024-2048-2048-1000", "batch": 4096,
     "optimizer": "adam", "precision": "bf16", "lr": 1e-4, "steps": 64},
    # One hidden layer of a wide bf16 model, forward.
    {"name": "linear_fwd_bf16", "kind": "linear", "op": "forward", "dtype": "bf16", "rows": 4096, "din": 4096,
     "dout": 4096},
    # The Linear 4096 -> 4096 backward at batch 8192: the largest products.
    {"name": "linear_bwd_bf16", "kind": "linear", "op": "backward", "dtype": "bf16", "rows": 8192, "din": 4096,
     "dout": 4096},
    # A hidden layer whose batch and widths are not multiples of any tile (the last batch of an epoch, a feature count
    # that the data set gave).
    {"name": "layer_bf16_ragged", "kind": "linear", "op": "layer", "dtype": "bf16", "rows": 4100, "din": 4000,
     "dout": 1000},
    # The same in f32, with odd widths: no row but the first is 16-byte aligned.
    {"name": "layer_f32_odd", "kind": "linear", "op": "layer", "dtype": "f32", "rows": 1500, "din": 1003, "dout": 777},
    # The tall-skinny weight gradient: dW and db over 262144 rows.
    {"name": "splitk_f16", "kind": "splitk", "dtype": "f16", "k": 262144, "m": 512, "n": 512, "slices": 64},
    # The tape's own benchmark: an epoch of 16 minibatches of 256 rows, as much host work as device work.
    {"name": "tape_relu_b256", "kind": "tape", "dims": "128-512-512-10", "act": "relu", "batch": 256, "batches": 16},
    # A model that only the tape can train (tanh layers, node by node), at a large batch and many classes.
    {"name": "tape_tanh_b2048", "kind": "tape", "dims": "512-1024-1024-1000", "act": "tanh", "batch": 2048,
     "batches": 4},
    # The softmax node over a wide head.
    {"name": "softmax_4096x1000", "kind": "softmax", "rows": 4096, "cols": 1000},
    # The optimizer alone over four 4096-wide layers.
    {"name": "adam_67m", "kind": "adam", "tensors": 4, "rows": 4096, "cols": 4096},
]


def listed():
    return [dict(c) for c in _LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A size of the range: half of them multiples of 64 (as layers are mostly chosen), the others any number."""
    n = _log(rng, lo, hi)
    return max(64, (n + 32) // 64 * 64) if rng.random() < 0.5 and hi >= 64 else n


def draw(rng):
    kind = rng.choice(["train", "train", "linear", "linear", "linear", "linear", "splitk", "tape", "softmax", "adam"])
    if kind == "train":
        dims = [_width(rng, 16, 1024) for _ in range(rng.randint(2, 4))] + [_log(rng, 2, 1000)]
        precision = rng.choice(["f32", "bf16"])
        optimizer = rng.choice(["adam", "sgd", "momentum"])
        lr = {"adam": 1e-3 if precision == "f32" else 1e-4, "sgd": 0.01, "momentum": 1e-3}[optimizer]
        return {"kind": kind, "dims": "-".join(map(str, dims)), "batch": _width(rng, 1, 4096), "optimizer": optimizer,
                "precision": precision, "lr": lr, "steps": rng.randint(16, 48)}
    if kind == "linear":
        dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
        most = 2048 if dtype == "f32" else 4096
        return {"kind": kind, "op": rng.choice(["forward", "backward", "layer"]), "dtype": dtype,
                "rows": _width(rng, 1, most), "din": _width(rng, 16, most), "dout": _width(rng, 10, most)}
    if kind == "splitk":
        m, n, k = _width(rng, 32, 512), _width(rng, 10, 512), _width(rng, 4096, 262144)
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "f16"]), "k": k, "m": m, "n": n,
                "slices": rng.choice([8, 16, 32, 64])}
    if kind == "tape":
        dims = [_width(rng, 16, 1024) for _ in range(rng.randint(2, 3))] + [_log(rng, 2, 1000)]
        return {"kind": kind, "dims": "-".join(map(str, dims)), "act": rng.choice(["relu", "tanh", "sigmoid"]),
                "batch": _width(rng, 16, 2048), "batches": rng.randint(2, 8)}
    if kind == "softmax":
        return {"kind": kind, "rows": _log(rng, 1, 16384), "cols": _log(rng, 2, 4096)}
    return {"kind": kind, "tensors": rng.randint(1, 12), "rows": _width(rng, 1, 2048), "cols": _width(rng, 16, 2048)}


# ------------------------------------------------------------------ device buffers

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_CODE = {"f32": G.F32, "bf16": G.BF16, "f16": G.F16}
_device = []


def _gpu():
    """The program's one context."""
    if not _device:
        _device.append(G.Gpu(0))
    return _device[0]


class _Window:
    """The device memory of a GpuTensor for torch, without a copy; keeps its owner alive.  A handle is a pointer to the
    buffer's record, which begins with its device pointer."""

    def __init__(self, t):
        self.owner = t
        kind = {G.F32: "<f4", G.BF16: "<i2", G.F16: "<f2", G.U32: "<i4"}[t.dtype]
        ptr = ctypes.c_void_p.from_address(t.handle).value
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": kind, "data": (ptr, False), "version": 3,
                                         "strides": None}


def _view(t):
    v = torch.as_tensor(_Window(t), device="cuda")
    return v.view(torch.bfloat16) if t.dtype == G.BF16 else v


def _buffer(shape, dtype="f32"):
    return _gpu().empty(tuple(shape), _CODE[dtype])


def _put(value, dtype="f32"):
    """A device buffer of these values, rounded to its type."""
    t = _buffer(value.shape, dtype)
    _view(t).copy_(value)
    return t


def _labels(value):
    t = _gpu().empty(tuple(value.shape), G.U32)
    _view(t).copy_(value.to(torch.int32))
    return t


# ------------------------------------------------------------------ inputs (from the seed alone)

def _dims(case):
    return [int(d) for d in case["dims"].split("-")]


def _normal(gen, shape, scale=1.0):
    return torch.randn(shape, generator=gen, device="cuda") * scale


def _uniform(gen, shape, bound):
    return (torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * bound


def _kaiming(gen, din, dout):
    return _uniform(gen, (din, dout), math.sqrt(6.0 / din))


def _inputs(case, seed):
    """The values that prepare() lays out and exact() computes with, on the GPU, already rounded to the types they are
    held in."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    kind = case["kind"]
    if kind in ("train", "tape"):
        dims, batch = _dims(case), case["batch"]
        n = case["steps"] if kind == "train" else case["batches"]
        params = []
        for a, b in zip(dims, dims[1:]):
            w = _kaiming(gen, a, b) if kind == "train" else _uniform(gen, (a, b), math.sqrt(6.0 / (a + b)))
            params += [w, _uniform(gen, (1, b), 1.0 / math.sqrt(a))]  # biases as of a network that has been trained
        half = kind == "train" and case["precision"] == "bf16"
        xs = []
        for _ in range(n):
            x = _normal(gen, (batch, dims[0]))
            xs.append(x.bfloat16() if half else x)
        ys = [torch.randint(0, dims[-1], (batch,), generator=gen, device="cuda") for _ in range(n)]
        return {"params": params, "x": xs, "y": ys}
    if kind == "linear":
        t, rows, din, dout = _TORCH[case["dtype"]], case["rows"], case["din"], case["dout"]
        x = _normal(gen, (rows, din))
        if case["op"] == "layer":  # the layer below ends in a ReLU
            x = x.relu()
        elif case["op"] == "backward":
            x = x / 64
        return {"x": x.to(t), "w": _kaiming(gen, din, dout).to(t), "b": _normal(gen, (1, dout), 0.1),
                "dy": _normal(gen, (rows, dout), 1 / 64).to(t)}
    if kind == "splitk":
        t = _TORCH[case["dtype"]]
        return {"x": _normal(gen, (case["k"], case["m"]), 1 / 16).to(t),
                "dy": _normal(gen, (case["k"], case["n"]), 1 / 16).to(t)}
    shape = (case["rows"], case["cols"])
    if kind == "softmax":
        return {"z": _normal(gen, shape, 3.0), "g": _normal(gen, shape)}
    each = []
    for _ in range(case["tensors"]):
        each.append({"theta": _uniform(gen, shape, 0.05), "g": _normal(gen, shape, 1e-3),
                     "m": _normal(gen, shape, 1e-3), "v": _normal(gen, shape, 1e-3).square()})
    return {"each": each}


_ADAM = {"lr": 1e-3, "betas": (0.9, 0.999), "eps": 1e-8}


def prepare(case, seed):
    gpu, kind, v = _gpu(), case["kind"], _inputs(case, seed)
    s = {"case": case}
    if kind == "train":
        sgd = case["optimizer"] != "adam"
        s["mlp"] = G.GpuMlp.from_params(gpu, [p.cpu().numpy() for p in v["params"]], case["batch"], case["lr"],
                                        optimizer="sgd" if sgd else "adam",
                                        momentum=0.9 if case["optimizer"] == "momentum" else 0.0,
                                        precision=case["precision"],
                                        loss_scale=1024.0 if case["precision"] == "bf16" else 1.0)
        s["batches"] = [(_put(x, case["precision"]), _labels(y)) for x, y in zip(v["x"], v["y"])]
    elif kind == "tape":
        dims = _dims(case)
        acts = [case["act"]] * (len(dims) - 2) + ["linear"]
        values = [p.cpu().numpy() for p in v["params"]]
        s["model"] = A.Sequential([A.Dense(gpu, dims[l], dims[l + 1], acts[l], weights=values[2 * l],
                                           bias=values[2 * l + 1]) for l in range(len(acts))])
        s["params"] = s["model"].params()
        s["opt"] = A.Adam(1e-3)
        s["batches"] = [(_put(x), _put(torch.nn.functional.one_hot(y, dims[-1]).float()))
                        for x, y in zip(v["x"], v["y"])]
        s["out"] = [_view(p.tensor) for p in s["params"]]
    elif kind == "linear":
        dtype, rows, din, dout = case["dtype"], case["rows"], case["din"], case["dout"]
        wide = "bf16" if dtype == "bf16" else "f32"  # what activations and their gradients are written as
        s.update(x=_put(v["x"], dtype), w=_put(v["w"], dtype), b=_put(v["b"]), dy=_put(v["dy"], dtype))
        out = {}
        if case["op"] != "backward":
            out["y"] = s["y"] = _buffer((rows, dout), wide)
        if case["op"] != "forward":
            out["dx"] = s["dx"] = _buffer((rows, din), wide)
            out["dw"] = s["dw"] = _buffer((din, dout))
            out["db"] = s["db"] = _buffer((1, dout))
        if case["op"] == "layer":  # the ReLU mask is the layer's input (f16 masks are not taken: its f32 values)
            s["mask"] = s["x"] if dtype != "f16" else _put(v["x"].float())
        s["out"] = {k: _view(t) for k, t in out.items()}
    elif kind == "splitk":
        m, n = case["m"], case["n"]
        s.update(x=_put(v["x"], case["dtype"]), dy=_put(v["dy"], case["dtype"]), dw=_buffer((m, n)), db=_buffer((1, n)),
                 part=_buffer((case["slices"] * (m * n + n),)))
        s["out"] = {"dw": _view(s["dw"]), "db": _view(s["db"])}
    elif kind == "softmax":
        s.update(z=_put(v["z"]), g=_put(v["g"]), p=_buffer(v["z"].shape), dz=_buffer(v["z"].shape))
        s["out"] = {"p": _view(s["p"]), "dz": _view(s["dz"])}
    else:
        s["t"] = 10  # updates applied so far
        for key in ("theta", "m", "v", "g"):
            s[key] = [_put(e[key]) for e in v["each"]]
        s["out"] = {key: [_view(t) for t in s[key]] for key in ("theta", "m", "v")}
    torch.cuda.synchronize()
    return s


def run(s):
    case, gpu = s["case"], _gpu()
    kind = case["kind"]
    if kind == "train":
        mlp = s["mlp"]
        for x, y in s["batches"]:
            mlp.step(x, y)
        return {"loss": mlp.last_loss(), "weights": mlp.weights()}
    if kind == "tape":
        loss = None
        for x, y in s["batches"]:
            tape = A.Tape(gpu)
            loss = A.softmax_cross_entropy(s["model"].forward(tape.constant(x)), y)
            s["opt"].step(s["params"], loss.backward())
        return {"loss": loss.item(), "weights": s["out"]}
    if kind == "linear":
        op = case["op"]
        if op != "backward":
            gpu.matmul_bias(s["x"], s["w"], s["y"], s["b"], True)
        if op == "backward":
            gpu.linear_backward(s["x"], s["dy"], s["w"], s["dx"], s["dw"], s["db"])
        elif op == "layer":
            gpu.matmul_at_b(s["x"], s["dy"], s["dw"], colsum=s["db"])
            gpu.matmul_a_bt(s["dy"], s["w"], s["dx"], relu_mask_from=s["mask"])
    elif kind == "splitk":
        gpu.split_k(s["x"], s["dy"], s["dw"], s["part"], case["slices"], True, colsum=s["db"])
    elif kind == "softmax":
        gpu.softmax_rows(s["z"], s["p"])
        gpu.softmax_rows_vjp(s["p"], s["g"], s["dz"])
    else:
        s["t"] += 1
        gpu.adam_many(s["theta"], s["m"], s["v"], s["g"], _ADAM["lr"], _ADAM["betas"], s["t"], _ADAM["eps"])
    return s["out"]


# ------------------------------------------------------------------ work

def work(case):
    kind = case["kind"]
    if kind in ("train", "tape"):
        dims, batch = _dims(case), case["batch"]
        n = case["steps"] if kind == "train" else case["batches"]
        mk = [a * b for a, b in zip(dims, dims[1:])]
        params = sum(mk) + sum(dims[1:])
        # Forward and dW of every layer, dX of all but the first.
        flops = 2 * batch * sum((3 if l else 2) * p for l, p in enumerate(mk))
        # The batch in; parameters, gradients and optimizer state as one update reads and writes them.
        state = {"adam": 28, "momentum": 20, "sgd": 12}[case.get("optimizer", "adam")]
        x = batch * dims[0] * (2 if case.get("precision") == "bf16" else 4)
        return {"bytes": n * (x + 4 * batch + state * params), "flops": n * flops}
    if kind == "linear":
        rows, din, dout = case["rows"], case["din"], case["dout"]
        i = 4 if case["dtype"] == "f32" else 2
        o = 2 if case["dtype"] == "bf16" else 4
        one = 2.0 * rows * din * dout
        fwd = i * (rows * din + din * dout) + 4 * dout + o * rows * dout
        bwd = i * (rows * din + rows * dout + din * dout) + o * rows * din + 4 * (din * dout + dout)
        if case["op"] == "forward":
            return {"bytes": fwd, "flops": one}
        if case["op"] == "backward":
            return {"bytes": bwd, "flops": 2 * one}
        # x and w are read once for both directions.
        return {"bytes": fwd + bwd - i * (rows * din + din * dout), "flops": 3 * one}
    if kind == "splitk":
        i = 4 if case["dtype"] == "f32" else 2
        k, m, n = case["k"], case["m"], case["n"]
        return {"bytes": i * k * (m + n) + 4 * (m * n + n), "flops": 2.0 * k * m * n}
    size = case["rows"] * case["cols"]
    if kind == "softmax":
        return {"bytes": 16 * size, "flops": 10 * size}  # z and g in, p and dz out
    return {"bytes": 28 * size * case["tensors"], "flops": 12 * size * case["tensors"]}


# ------------------------------------------------------------------ 64-bit results

def _train_exact(case, v, adam, acts):
    """The training loop in 64 bits: (last loss, parameters)."""
    ps = [p.double() for p in v["params"]]
    m, w2 = [torch.zeros_like(p) for p in ps], [torch.zeros_like(p) for p in ps]
    momentum = 0.9 if case.get("optimizer") == "momentum" else 0.0
    loss, lr = None, case.get("lr", 1e-3)
    layers = len(ps) // 2
    for t, (x, y) in enumerate(zip(v["x"], v["y"]), 1):
        a = [x.double()]
        for l in range(layers):
            z = a[-1] @ ps[2 * l] + ps[2 * l + 1]
            a.append(z if l == layers - 1 else {"relu": torch.relu, "tanh": torch.tanh, "sigmoid": torch.sigmoid}[acts](z))
        p = torch.softmax(a[-1], dim=1)
        rows = torch.arange(len(y), device=y.device)
        loss = -p[rows, y].clamp_min(1e-12).log().mean()
        p[rows, y] -= 1.0
        d = p / len(y)
        grads = [None] * len(ps)
        for l in range(layers - 1, -1, -1):
            grads[2 * l], grads[2 * l + 1] = a[l].T @ d, d.sum(0, keepdim=True)
            if l:
                d = d @ ps[2 * l].T
                h = a[l]
                d = d * {"relu": (h > 0).double(), "tanh": 1 - h * h, "sigmoid": h * (1 - h)}[acts]
        for i, g in enumerate(grads):
            if adam:
                m[i] = 0.9 * m[i] + 0.1 * g
                w2[i] = 0.999 * w2[i] + 0.001 * g * g
                ps[i] = ps[i] - lr * (m[i] / (1 - 0.9 ** t)) / ((w2[i] / (1 - 0.999 ** t)).sqrt() + 1e-8)
            else:
                m[i] = momentum * m[i] + lr * g
                ps[i] = ps[i] - m[i]
    return float(loss), ps


def exact(case, seed):
    kind, v = case["kind"], _inputs(case, seed)
    if kind == "train":
        loss, ps = _train_exact(case, v, case["optimizer"] == "adam", "relu")
        return {"loss": loss, "weights": ps}
    if kind == "tape":
        loss, ps = _train_exact(case, v, True, case["act"])
        return {"loss": loss, "weights": ps}
    if kind == "linear":
        x, w, b, dy = (v[k].double() for k in ("x", "w", "b", "dy"))
        out = {}
        if case["op"] != "backward":
            out["y"] = torch.relu(x @ w + b)
        if case["op"] != "forward":
            dx = dy @ w.T
            out["dx"] = dx * (x > 0) if case["op"] == "layer" else dx
            out["dw"], out["db"] = x.T @ dy, dy.sum(0, keepdim=True)
        return out
    if kind == "splitk":
        x, dy = v["x"].double(), v["dy"].double()
        return {"dw": x.T @ dy, "db": dy.sum(0, keepdim=True)}
    if kind == "softmax":
        p = torch.softmax(v["z"].double(), dim=1)
        g = v["g"].double()
        return {"p": p, "dz": p * (g - (g * p).sum(1, keepdim=True))}
    out = {"theta": [], "m": [], "v": []}
    (b1, b2), t = _ADAM["betas"], 11
    for e in v["each"]:
        th, g, m, w2 = (e[k].double() for k in ("theta", "g", "m", "v"))
        m, w2 = b1 * m + (1 - b1) * g, b2 * w2 + (1 - b2) * g * g
        out["m"].append(m)
        out["v"].append(w2)
        out["theta"].append(th - _ADAM["lr"] * (m / (1 - b1 ** t)) / ((w2 / (1 - b2 ** t)).sqrt() + _ADAM["eps"]))
    return out


def tolerance(case):
    kind = case["kind"]
    if kind == "train":
        # Against 64 bits the weights are up to 5e-3 off after 32 f32 Adam steps (gradients near zero change sign, and
        # Adam divides by their size), up to 5e-5 after 200 f32 SGD steps, and 3e-3 to 8e-3 off in bf16.
        if case["precision"] == "bf16":
            return {"rel": 0.02, "max": 0.5}
        return {"rel": 0.02, "max": 0.6} if case["optimizer"] == "adam" else {"rel": 4e-4, "max": 2e-2}
    if kind == "tape":  # Adam again: 5e-6 (tanh) to 8e-4 (ReLU) off
        return {"rel": 4e-3, "max": 0.3}
    if kind in ("linear", "splitk"):
        # f32 sums in another order (1e-7 to 7e-7 off); a bf16 result is rounded once more (2e-3).
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 4e-6}
    return {"rel": 4e-6}  # 1e-7 to 9e-7 off
