"""The calls that a user of this backend has it do, as cases that can be timed and compared.

Everything goes through the C ABI of include/kd_api.h (kael.cpp_amd/kd.py): device buffers are torch
tensors on the default stream, which is the backend's own. A training step is the list of calls that
kael's training loop issues for it with its optional device branches, each argument built once, as a
program that runs the same step over and over holds them.

Sizes are those of the repository's configurations (C1-C5: the 512 and 4096 products, the 4096 x 4096
elementwise set, the 784-128-10 MLP, the char-level GPT, GPT-2 small) and of its bench sections, with
ragged ones among them; `draw` spreads each kind over its whole range.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "kael.cpp_amd"))
import kd  # noqa: E402

GPT2 = {"vocab": 50257, "positions": 1024, "layers": 12, "heads": 12}  # GPT-2 small: heads of 64
TORCH = {"f32": torch.float32, "f64": torch.float64}
KD = {"f32": kd.F32, "f64": kd.F64}
EPS = 1e-5


def listed():
    return [
        # C3: one SGD step of the image MLP. The smallest calls: every kernel is a few microseconds, so
        # launches and the range check's round trip decide.
        {"name": "mlp_step_784_128_10", "kind": "mlp_step", "batch": 64, "inputs": 784, "hidden": 128, "classes": 10},
        # C1: one small square product.
        {"name": "matmul_512", "kind": "matmul", "batches": 1, "rows": 512, "inner": 512, "columns": 512,
         "dtype": "f32"},
        # The headline: one large square product.
        {"name": "matmul_4096", "kind": "matmul", "batches": 1, "rows": 4096, "inner": 4096, "columns": 4096,
         "dtype": "f32"},
        # GPT-2 small's attention over full contexts, forward and backward.
        {"name": "attention_8x1024x12", "kind": "attention", "batch": 8, "length": 1024, "heads": 12},
        # C4: one whole training step (forward, backward, Adam) of the char-level GPT.
        {"name": "gpt_step_char", "kind": "gpt_step", "batch": 32, "length": 128, "layers": 4, "heads": 4,
         "vocab": 96, "positions": 128},
        # A training step of two GPT-2 small layers with GPT-2's vocabulary over ragged sequences: the
        # products, the loss rows and the optimizer at GPT-2's widths.
        {"name": "gpt_step_wide_ragged", "kind": "gpt_step", "batch": 3, "length": 333, "layers": 2, "heads": 12,
         "vocab": 50257, "positions": 1024},
        # A long prompt through GPT-2 small, of a length that no tile divides.
        {"name": "prefill_1000", "kind": "prefill", "prompt": 1000},
        # C5: GPT-2 small generating greedily from a 64-token prompt.
        {"name": "decode_greedy_64", "kind": "decode", "prompt": 64, "tokens": 64, "temperature": 0.0, "top_k": 0},
        # kael's default generation: temperature 1 over the whole vocabulary.
        {"name": "decode_sampled_16", "kind": "decode", "prompt": 64, "tokens": 16, "temperature": 1.0, "top_k": 0},
        # C2: broadcasting and transposed elementwise work on one matrix, and its reductions and scans.
        {"name": "tensor_ops_4096", "kind": "tensor_ops", "rows": 4096, "columns": 4096, "dtype": "f32"},
        # The row kernels and their backward passes over a large activation.
        {"name": "rows_32768x1024", "kind": "rows", "rows": 32768, "columns": 1024, "dtype": "f32"},
        # Dropout of the char-level GPT's activations with kael's own random stream.
        {"name": "dropout_32x128x256", "kind": "dropout", "count": 32 * 128 * 256, "keep": 0.9, "dtype": "f32"},
    ]


def draw(rng):
    def log_int(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    def size(low, high):  # as often a multiple of 64 or 4 as any number
        unit = rng.choice((1, 1, 4, 64))
        return max(low, log_int(low, high) // unit * unit)

    largest = max(cost(c) for c in listed())
    while True:
        kind = rng.choice(("mlp_step", "matmul", "matmul", "attention", "gpt_step", "gpt_step", "prefill", "decode",
                           "tensor_ops", "rows", "dropout"))
        dtype = "f64" if rng.random() < 0.2 else "f32"
        if kind == "mlp_step":
            case = {"batch": log_int(1, 1024), "inputs": size(16, 3072), "hidden": size(16, 1024),
                    "classes": log_int(2, 100)}
        elif kind == "matmul":
            case = {"batches": rng.choice((1, 1, 1, log_int(2, 32))), "rows": size(16, 4096), "inner": size(16, 4096),
                    "columns": size(16, 4096), "dtype": dtype}
            if 2.0 * case["batches"] * case["rows"] * case["inner"] * case["columns"] > 2.0 * 4096 ** 3:
                continue
        elif kind == "attention":
            case = {"batch": log_int(1, 32), "length": log_int(1, 1024), "heads": rng.randint(1, 16)}
            if case["batch"] * case["length"] > 8192:
                continue
        elif kind == "gpt_step":
            length = log_int(8, 512)
            case = {"batch": log_int(1, 64), "length": length, "layers": rng.randint(1, 4),
                    "heads": rng.randint(1, 12), "vocab": log_int(50, 50257), "positions": length + rng.randint(0, 100)}
            if case["batch"] * length > 4096:
                continue
        elif kind == "prefill":
            case = {"prompt": log_int(1, 1024)}
        elif kind == "decode":
            temperature = rng.choice((0.0, 0.8, 1.0))
            case = {"prompt": log_int(1, 900), "tokens": log_int(8, 64), "temperature": temperature,
                    "top_k": rng.choice((0, 40)) if temperature else 0}
            if temperature and not case["top_k"]:
                case["tokens"] = min(case["tokens"], 16)
        elif kind == "tensor_ops":
            case = {"rows": size(16, 4096), "columns": size(16, 4096), "dtype": dtype}
        elif kind == "rows":
            case = {"rows": log_int(1, 32768), "columns": size(16, 4096), "dtype": dtype}
            if case["rows"] * case["columns"] * (2 if dtype == "f64" else 1) > 32768 * 1024:
                continue
        else:
            case = {"count": log_int(100, 1 << 22), "keep": rng.choice((0.5, 0.8, 0.9, 0.95)), "dtype": dtype}
        case["kind"] = kind
        if cost(case) <= largest:
            return case


def cost(case):
    done = work(case)
    return max(done["bytes"], done["flops"] / 50)


# ---- the calls ------------------------------------------------------------------------------------


def backend():
    return kd.load()


def ptr(tensor):
    return ctypes.c_void_p(tensor.data_ptr())


class Calls:
    """A list of C ABI calls with their arguments, and the tensors that they use."""

    def __init__(self):
        self.steps, self.held = [], []

    def add(self, name, *args):
        given = []
        for a in args:
            if isinstance(a, torch.Tensor):
                self.held.append(a)
                a = ptr(a)
            elif isinstance(a, ctypes.Structure) and not isinstance(a, kd.ElementParameters):
                self.held.append(a)
                a = ctypes.byref(a)
            given.append(a)
        self.steps.append((getattr(backend().lib, "kd_" + name), tuple(given), name))

    def run(self):
        for call, args, name in self.steps:
            rc = call(*args)
            if rc:
                backend().check(rc, "kd_" + name)

    def element(self, op, shape, *operands):
        """One elementwise call; an operand is (tensor, element strides over `shape`)."""
        size = operands[1][0].element_size()
        layout = kd.element_layout(shape, [tuple(s * t.element_size() for s in strides) for t, strides in operands],
                                   [t.data_ptr() for t, _ in operands])
        self.held += [t for t, _ in operands]
        dtype = kd.F32 if size == 4 else kd.F64
        self.add("elementwise", kd.OP[op], dtype, dtype, layout, kd.params())

    def flat(self, op, *tensors):
        """The same over contiguous tensors of one size; a tensor of one element is a scalar."""
        n = tensors[0].numel()
        self.element(op, (n,), *((t, (1 if t.numel() == n else 0,)) for t in tensors))

    def product(self, out, a, b, rows, inner, columns, a_by=None, b_by=None, bias=None):
        """out [rows, columns] = a . b, each operand's (row, column) strides as given or row-major."""
        strides = kd.MatmulStrides((0, *(a_by or (inner, 1))), (0, *(b_by or (columns, 1))), (0, columns, 1))
        args = (kd.F32, a, b, out, kd.MatmulSizes(1, rows, inner, columns), strides)
        if bias is None:
            self.add("matmul_strided", *args)
        else:
            self.add("matmul_strided_bias", *args, bias)

    def linear(self, out, x, weight, bias):
        """out = x . weight^T + bias, weight [out features, in features]."""
        rows, (columns, inner) = x.numel() // weight.shape[1], weight.shape
        self.product(out, x, weight, rows, inner, columns, b_by=(1, inner), bias=bias)

    def linear_backward(self, grad, x, weight, grad_x, grad_weight, grad_bias):
        columns, inner = weight.shape
        rows = x.numel() // inner
        if grad_bias is not None:
            self.add("reduce_columns", kd.REDUCE_SUM, kd.F32, kd.F32, grad_bias, grad, rows, columns)
        if grad_x is not None:
            self.product(grad_x, grad, weight, rows, columns, inner)
        self.product(grad_weight, grad, x, columns, rows, inner, a_by=(1, columns))

    def loss(self, logits, targets, grad, row_loss, mean, count, weights):
        """Mean cross-entropy of the rows and its gradient, after the range check of the targets."""
        rows, columns = logits.shape
        bounds = np.zeros(2, np.int64)
        self.held.append(bounds)
        self.add("index_bounds", targets, rows, 1, bounds.ctypes.data_as(ctypes.c_void_p))
        self.add("cross_entropy_rows", kd.F32, row_loss, logits, targets, rows, columns)
        self.add("reduce", kd.REDUCE_SUM, kd.F32, kd.F32, mean, row_loss, rows, 1)
        self.flat("DIVIDES", mean, mean, count)
        self.add("cross_entropy_grad", kd.F32, grad, logits, targets, weights, rows, columns)


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def uniform(gen, shape, low, high, dtype=torch.float32):
    return torch.rand(shape, generator=gen, device="cuda", dtype=dtype) * (high - low) + low


def normal(gen, shape, deviation, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype) * deviation


def whole(gen, shape, high):
    return torch.randint(0, high, shape, generator=gen, device="cuda")


def empty(*shape, dtype=torch.float32):
    return torch.empty(shape, device="cuda", dtype=dtype)


def inputs(case, seed):
    """The tensors that a case starts from, by name: what the backend and `exact` both see."""
    gen, kind = generator(seed), case["kind"]
    dtype = TORCH.get(case.get("dtype"))
    if kind == "mlp_step":
        given = {"x": uniform(gen, (case["batch"], case["inputs"]), 0, 1),
                 "targets": whole(gen, (case["batch"],), case["classes"])}
        for name, fan, features in (("1", case["inputs"], case["hidden"]), ("2", case["hidden"], case["classes"])):
            given["w" + name] = uniform(gen, (features, fan), -fan ** -0.5, fan ** -0.5)
            given["b" + name] = uniform(gen, (features,), -fan ** -0.5, fan ** -0.5)
        return given
    if kind == "matmul":
        return {"a": uniform(gen, (case["batches"], case["rows"], case["inner"]), -1, 1, dtype),
                "b": uniform(gen, (case["batches"], case["inner"], case["columns"]), -1, 1, dtype)}
    if kind == "attention":
        features = case["heads"] * 64
        return {"qkv": normal(gen, (case["batch"], case["length"], 3, case["heads"], 64), 1.0),
                "grad": normal(gen, (case["batch"], case["length"], features), 1.0)}
    if kind == "gpt_step":
        return {"tokens": whole(gen, (case["batch"], case["length"]), case["vocab"]),
                "targets": whole(gen, (case["batch"], case["length"]), case["vocab"]),
                "weights": gpt_weights(gen, case)}
    if kind in ("prefill", "decode"):
        given = {"weights": gpt_weights(gen, GPT2), "prompt": whole(gen, (case["prompt"],), GPT2["vocab"])}
        if kind == "decode":
            given["uniforms"] = uniform(gen, (case["tokens"],), 0, 1, torch.float64)
        return given
    if kind == "tensor_ops":
        return {"a": uniform(gen, (case["rows"], case["columns"]), -1, 1, dtype),
                "b": uniform(gen, (case["rows"],), -1, 1, dtype),
                "c": uniform(gen, (case["columns"], case["rows"]), -1, 1, dtype)}
    if kind == "rows":
        shape, columns = (case["rows"], case["columns"]), case["columns"]
        return {"x": normal(gen, shape, 1.0, dtype), "grad": normal(gen, shape, 1.0, dtype),
                "weight": 1 + normal(gen, (columns,), 0.1, dtype), "bias": normal(gen, (columns,), 0.1, dtype)}
    return {"x": normal(gen, (case["count"],), 1.0, dtype)}


def gpt_weights(gen, case):
    """The GPT's parameters by kael's names: N(0, 0.02), LayerNorm gain 1 and bias 0, as C4 and C5 have them."""
    weights = {}
    for name, shape in kd.gpt2_parameter_shapes(case["vocab"], case["positions"], case["layers"], case["heads"] * 64):
        if ".ln" in name or name.startswith("ln"):
            weights[name] = torch.full(shape, float(name.endswith("weight")), device="cuda")
        else:
            weights[name] = normal(gen, shape, 0.02)
    return weights


def prepare(case, seed):
    given = inputs(case, seed)
    return {"case": case, "calls": Calls(), "out": {}, **globals()["prepare_" + case["kind"]](case, seed, given)}


def run(state):
    kind = state["case"]["kind"]
    if kind in ("prefill", "decode"):
        engine = state["engine"]
        if state["case"].get("temperature"):
            engine.set_uniforms(state["uniforms"])
        engine.prefill(state["prompt"])
        if kind == "prefill":
            return {"logits": engine.logits()}
        engine.decode(state["case"]["tokens"] - 1)
        return {"tokens": engine.sequence(), "logits": engine.logits()}
    state["calls"].run()
    return state["out"]


def prepare_matmul(case, seed, given):
    calls, dtype = Calls(), case["dtype"]
    out = empty(case["batches"], case["rows"], case["columns"], dtype=TORCH[dtype])
    calls.add("matmul", KD[dtype], given["a"], given["b"], out,
              kd.MatmulSizes(case["batches"], case["rows"], case["inner"], case["columns"]))
    return {"calls": calls, "out": {"product": out}}


def prepare_mlp_step(case, seed, given):
    calls = Calls()
    batch, hidden, classes = case["batch"], case["hidden"], case["classes"]
    x, targets, w1, b1, w2, b2 = (given[n] for n in ("x", "targets", "w1", "b1", "w2", "b2"))
    z, h, dh, mask, logits, dlogits = (empty(batch, n) for n in (hidden, hidden, hidden, hidden, classes, classes))
    positive = empty(batch, hidden, dtype=torch.uint8)
    row_loss, mean = empty(batch), empty(1)
    grads = {n: torch.empty_like(given[n]) for n in ("w1", "b1", "w2", "b2")}
    zero, count = torch.zeros(1, device="cuda"), torch.full((1,), float(batch), device="cuda")
    calls.linear(z, x, w1, b1)
    calls.flat("RELU", h, z)
    calls.linear(logits, h, w2, b2)
    calls.loss(logits, targets, dlogits, row_loss, mean, count, torch.full((batch,), 1.0 / batch, device="cuda"))
    calls.linear_backward(dlogits, h, w2, dh, grads["w2"], grads["b2"])
    calls.flat("GREATER", positive, z, zero)
    layout = kd.element_layout((mask.numel(),), [(4,), (1,)], [mask.data_ptr(), positive.data_ptr()])
    calls.held += [mask, positive]
    calls.add("convert", kd.F32, kd.BOOL, layout)
    calls.flat("TIMES", dh, dh, mask)
    calls.linear_backward(dh, x, w1, None, grads["w1"], grads["b1"])
    for n in ("w1", "b1", "w2", "b2"):
        calls.add("sgd_step", kd.F32, given[n], grads[n], given[n].numel(), 0.01, 0.0)
    return {"calls": calls, "out": {"loss": mean, "logits": logits, "grads": grads,
                                    "updated": {n: given[n] for n in grads}}}


def prepare_attention(case, seed, given):
    calls, qkv, grad = Calls(), given["qkv"], given["grad"]
    sizes = (case["batch"], case["length"], case["heads"], 64)
    out, lse, dqkv = torch.empty_like(grad), empty(case["batch"], case["heads"], case["length"]), torch.empty_like(qkv)
    calls.add("causal_attention", kd.F32, out, lse, qkv, *sizes)
    calls.add("causal_attention_backward", kd.F32, dqkv, grad, qkv, out, lse, *sizes)
    return {"calls": calls, "out": {"out": out, "lse": lse, "dqkv": dqkv}}


def flat_views(shapes):
    """One zeroed buffer, and a view of it for each shape on a 256-byte boundary."""
    at, places = 0, {}
    for name, shape in shapes.items():
        n = math.prod(shape)
        places[name] = (at, n, shape)
        at += -(-n // 64) * 64
    flat = torch.zeros(at, device="cuda")
    return flat, {name: flat[a:a + n].view(shape) for name, (a, n, shape) in places.items()}


def adam_moments(weights, seed):
    """Moments as they stand in the middle of a run: first ones of either sign, second ones above their squares."""
    gen = generator(seed + 1)
    first = {n: normal(gen, w.shape, 1e-4) for n, w in weights.items()}
    return first, {n: m * m + 1e-6 for n, m in first.items()}


ADAM = {"lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8, "step": 100}


def prepare_gpt_step(case, seed, given):
    """Forward, loss, backward and Adam of kael's GPT in the calls that kael's own loop issues."""
    calls = Calls()
    batch, length, heads = case["batch"], case["length"], case["heads"]
    rows, d, vocab = batch * length, heads * 64, case["vocab"]
    flat, p = flat_views({n: tuple(w.shape) for n, w in given["weights"].items()})
    for n, w in given["weights"].items():
        p[n].copy_(w)
    _, g = flat_views({n: tuple(w.shape) for n, w in p.items()})
    first, second = adam_moments(given["weights"], seed)
    tokens, targets = given["tokens"], given["targets"]

    def new(columns=d):
        return empty(rows, columns)

    def norm(out, standardized, x, name):
        calls.add("layer_norm_rows", kd.F32, out, standardized, x, rows, d, EPS, p[name + ".weight"], p[name + ".bias"])

    def norm_backward(grad, x, standardized, name):
        dx = new()
        calls.add("layer_norm_rows_backward", kd.F32, dx, g[name + ".weight"], g[name + ".bias"], x, standardized, grad,
                  p[name + ".weight"], rows, d, EPS)
        return dx

    def linear(x, name):
        out = new(p[name + ".weight"].shape[0])
        calls.linear(out, x, p[name + ".weight"], p[name + ".bias"])
        return out

    def linear_backward(grad, x, name):
        dx = torch.empty_like(x)
        calls.linear_backward(grad, x, p[name + ".weight"], dx, g[name + ".weight"], g[name + ".bias"])
        return dx

    def add(a, b):
        out = new()
        calls.flat("PLUS", out, a, b)
        return out

    bounds = np.zeros(2, np.int64)
    calls.held.append(bounds)
    calls.add("index_bounds", tokens, rows, 1, bounds.ctypes.data_as(ctypes.c_void_p))
    embedded, x = new(), new()
    index = kd.index_layout((rows, d), 0, (d, 1), (1, 0), (d, 1))
    calls.add("gather", kd.F32, embedded, p["token_embedding.weight"], tokens, index)
    calls.element("PLUS", (batch, length * d), (x, (length * d, 1)), (embedded, (length * d, 1)),
                  (p["position_embedding.weight"], (0, 1)))
    kept = []
    for layer in range(case["layers"]):
        b = f"blocks.{layer}."
        n1, s1, n2, s2, out = new(), new(), new(), new(), new()
        lse = empty(batch, heads, length)
        norm(n1, s1, x, b + "ln1")
        qkv = linear(n1, b + "attn.qkv")
        calls.add("causal_attention", kd.F32, out, lse, qkv, batch, length, heads, 64)
        middle = add(x, linear(out, b + "attn.proj"))
        norm(n2, s2, middle, b + "ln2")
        z = linear(n2, b + "mlp.fc1")
        h = torch.empty_like(z)
        calls.flat("GELU_TANH", h, z)
        kept.append((x, n1, s1, qkv, lse, out, middle, n2, s2, z, h))
        x = add(middle, linear(h, b + "mlp.fc2"))
    last, standardized = new(), new()
    norm(last, standardized, x, "ln_final")
    logits, dlogits, row_loss, mean = new(vocab), new(vocab), empty(rows), empty(1)
    head = p["token_embedding.weight"]
    calls.product(logits, last, head, rows, d, vocab, b_by=(1, d))
    calls.loss(logits, targets, dlogits, row_loss, mean, torch.full((1,), float(rows), device="cuda"),
               torch.full((rows,), 1.0 / rows, device="cuda"))
    grad = new()
    calls.linear_backward(dlogits, last, head, grad, g["token_embedding.weight"], None)
    grad = norm_backward(grad, x, standardized, "ln_final")
    for layer in reversed(range(case["layers"])):
        b = f"blocks.{layer}."
        x, n1, s1, qkv, lse, out, middle, n2, s2, z, h = kept[layer]
        dh = linear_backward(grad, h, b + "mlp.fc2")
        dz, dqkv = torch.empty_like(z), torch.empty_like(qkv)
        calls.flat("GELU_TANH_BACKWARD", dz, z, dh)
        grad = add(grad, norm_backward(linear_backward(dz, n2, b + "mlp.fc1"), middle, s2, b + "ln2"))
        calls.add("causal_attention_backward", kd.F32, dqkv, linear_backward(grad, out, b + "attn.proj"), qkv, out, lse,
                  batch, length, heads, 64)
        grad = add(grad, norm_backward(linear_backward(dqkv, n1, b + "attn.qkv"), x, s1, b + "ln1"))
    calls.add("reduce_columns", kd.REDUCE_SUM, kd.F32, kd.F32, g["position_embedding.weight"], grad, batch, length * d)
    calls.add("scatter_add", kd.F32, g["token_embedding.weight"], tokens, grad, index)
    table = (kd.AdamTensor * len(p))(*(kd.AdamTensor(p[n].data_ptr(), g[n].data_ptr(), first[n].data_ptr(),
                                                     second[n].data_ptr(), p[n].numel(), ADAM["step"]) for n in p))
    calls.held += [table, *first.values(), *second.values(), flat]
    calls.add("adam_step_many", kd.F32, table, len(p), ADAM["lr"], ADAM["beta1"], ADAM["beta2"], ADAM["eps"], 0.0, 0)
    return {"calls": calls, "out": {"loss": mean, "grads": g, "updated": flat}}


def prepare_prefill(case, seed, given):
    engine = kd.Gpt(backend(), GPT2["vocab"], GPT2["positions"], GPT2["layers"], GPT2["heads"], GPT2["heads"] * 64)
    torch.cuda.synchronize()
    for name, w in given["weights"].items():
        backend().check(backend().lib.kd_gpt_load_parameter_device(engine.handle, name.encode(), ptr(w), w.numel()), name)
    return {"engine": engine, "prompt": given["prompt"].cpu().numpy()}


def prepare_decode(case, seed, given):
    state = prepare_prefill(case, seed, given)
    if case["temperature"]:
        state["engine"].set_sampling(case["temperature"], case["top_k"])
    return {**state, "uniforms": given["uniforms"].cpu().numpy()}


def prepare_tensor_ops(case, seed, given):
    calls, rows, columns, dtype = Calls(), case["rows"], case["columns"], KD[case["dtype"]]
    a, b, c = given["a"], given["b"], given["c"]
    like = torch.empty_like
    out = {"sum": like(a), "product": like(a), "transposed": like(c), "scan": like(a),
           "row_sum": empty(rows, dtype=a.dtype), "column_sum": empty(columns, dtype=a.dtype),
           "row_argmax": empty(rows, dtype=torch.int64), "largest": empty(1, dtype=a.dtype)}
    calls.element("PLUS", (rows, columns), (out["sum"], (columns, 1)), (a, (columns, 1)), (b, (1, 0)))
    calls.element("TIMES", (rows, columns), (out["product"], (columns, 1)), (a, (columns, 1)), (b, (1, 0)))
    calls.element("PLUS", (columns, rows), (out["transposed"], (rows, 1)), (a, (1, columns)), (c, (rows, 1)))
    calls.add("reduce", kd.REDUCE_SUM, dtype, dtype, out["row_sum"], a, columns, rows)
    calls.add("reduce_columns", kd.REDUCE_SUM, dtype, dtype, out["column_sum"], a, rows, columns)
    calls.add("arg_reduce", 1, dtype, out["row_argmax"], a, columns, rows)
    calls.add("cumsum", dtype, out["scan"], a, columns, rows)
    calls.add("reduce", kd.REDUCE_MAX, dtype, dtype, out["largest"], a, rows * columns, 1)
    return {"calls": calls, "out": out}


def prepare_rows(case, seed, given):
    calls, rows, columns, dtype = Calls(), case["rows"], case["columns"], KD[case["dtype"]]
    x, grad, weight, bias = (given[n] for n in ("x", "grad", "weight", "bias"))
    out = {n: torch.empty_like(x) for n in ("softmax", "softmax_dx", "norm", "standardized", "norm_dx", "gelu", "gelu_dx")}
    out.update({n: torch.empty_like(weight) for n in ("norm_dweight", "norm_dbias")})
    calls.add("softmax_rows", dtype, out["softmax"], x, rows, columns, 0)
    calls.add("softmax_rows_backward", dtype, out["softmax_dx"], out["softmax"], grad, rows, columns, 0)
    calls.add("layer_norm_rows", dtype, out["norm"], out["standardized"], x, rows, columns, EPS, weight, bias)
    calls.add("layer_norm_rows_backward", dtype, out["norm_dx"], out["norm_dweight"], out["norm_dbias"], x,
              out["standardized"], grad, weight, rows, columns, EPS)
    calls.flat("GELU_TANH", out["gelu"], x)
    calls.flat("GELU_TANH_BACKWARD", out["gelu_dx"], x, grad)
    return {"calls": calls, "out": out}


def prepare_dropout(case, seed, given):
    calls, x = Calls(), given["x"]
    state = np.zeros(313, np.uint64)
    backend().lib.kd_mt19937_64_seed(state.ctypes.data_as(ctypes.c_void_p), seed)
    out, mask = torch.empty_like(x), torch.empty_like(x)
    calls.held.append(state)
    calls.add("dropout", KD[case["dtype"]], out, mask, x, case["count"], case["keep"],
              state.ctypes.data_as(ctypes.c_void_p))
    return {"calls": calls, "out": {"out": out, "mask": mask, "generator": state.view(np.int64)}}


# ---- what they cannot do without --------------------------------------------------------------------


def gpt_parameters(case):
    return sum(math.prod(s) for _, s in kd.gpt2_parameter_shapes(case["vocab"], case["positions"], case["layers"],
                                                                 case["heads"] * 64))


def work(case):
    kind, item = case["kind"], 8 if case.get("dtype") == "f64" else 4
    if kind == "mlp_step":
        n, i, h, c = (case[k] for k in ("batch", "inputs", "hidden", "classes"))
        weights = i * h + h + h * c + c
        return {"bytes": 4 * (n * i + 3 * weights + n * c) + 8 * n, "flops": 2 * n * (2 * i * h + 3 * h * c)}
    if kind == "matmul":
        b, m, k, n = (case[k] for k in ("batches", "rows", "inner", "columns"))
        return {"bytes": item * b * (m * k + k * n + m * n), "flops": 2 * b * m * k * n}
    if kind == "attention":
        b, t, h = case["batch"], case["length"], case["heads"]
        # Two products forward and four backward over the unmasked pairs.
        return {"bytes": 4 * b * t * h * (64 * 8 + 1), "flops": 12 * 64 * b * h * (t * (t + 1) // 2)}
    if kind == "gpt_step":
        d, tokens = case["heads"] * 64, case["batch"] * case["length"]
        per_token = case["layers"] * 12 * d * d + d * case["vocab"]
        pairs = case["batch"] * case["heads"] * case["layers"] * case["length"] * (case["length"] + 1) // 2
        return {"bytes": 28 * gpt_parameters(case) + 16 * tokens, "flops": 6 * per_token * tokens + 12 * 64 * pairs}
    if kind in ("prefill", "decode"):
        d, layers, prompt, steps = 768, GPT2["layers"], case["prompt"], case.get("tokens", 1) - 1
        body, head = layers * 12 * d * d, d * GPT2["vocab"]
        context = sum(range(prompt + 1, prompt + steps + 1))
        pairs = prompt * (prompt + 1) // 2 + context
        return {"bytes": 4 * (body + head) * (1 + steps) + 8 * layers * d * context + 4 * GPT2["vocab"],
                "flops": 2 * body * (prompt + steps) + 2 * head * (1 + steps) + 4 * d * layers * pairs}
    if kind == "tensor_ops":
        r, c = case["rows"], case["columns"]
        return {"bytes": item * (6 * r * c + 2 * r + c) + 8 * r, "flops": 7 * r * c}
    if kind == "rows":
        r, c = case["rows"], case["columns"]
        return {"bytes": item * (9 * r * c + 4 * c), "flops": 60 * r * c}
    return {"bytes": 3 * item * case["count"], "flops": 2 * case["count"]}


def tolerance(case):
    # About four times what the results are off 64 bits, measured: another order of the same sums moves them by as
    # much. Sums over thousands of f32 products (matmul, the GPT's gradients through a vocabulary of 50257) are the
    # widest; elementwise results and sums held in 64 bits are off by their own rounding only.
    if case.get("dtype") == "f64":
        return {"rel": 1e-14 if case["kind"] == "dropout" else 1e-13}
    return {"rel": {"mlp_step": 1e-6, "matmul": 4e-6, "attention": 2e-6, "gpt_step": 2e-5, "prefill": 4e-6,
                    "decode": 4e-6, "tensor_ops": 2e-7, "rows": 4e-7, "dropout": 2e-7}[case["kind"]]}


# ---- the same in 64 bits ----------------------------------------------------------------------------


def exact(case, seed):
    return globals()["exact_" + case["kind"]](case, seed, inputs(case, seed))


def exact_matmul(case, seed, given):
    return {"product": torch.stack([a.double() @ b.double() for a, b in zip(given["a"], given["b"])])}


def exact_mlp_step(case, seed, given):
    p = {n: given[n].double().requires_grad_() for n in ("w1", "b1", "w2", "b2")}
    h = torch.relu(given["x"].double() @ p["w1"].t() + p["b1"])
    logits = h @ p["w2"].t() + p["b2"]
    loss = torch.nn.functional.cross_entropy(logits, given["targets"])
    grads = dict(zip(p, torch.autograd.grad(loss, list(p.values()))))
    return {"loss": loss.reshape(1), "logits": logits, "grads": grads,
            "updated": {n: p[n] - 0.01 * grads[n] for n in p}}


def attend(qkv):
    """Causal attention of qkv [B, T, 3, H, 64]: its output [B, T, H * 64] and each row's log-sum-exp."""
    b, t, _, h, _ = qkv.shape
    q, k, v = (qkv[:, :, i].transpose(1, 2).contiguous() for i in range(3))
    mask = torch.ones(t, t, dtype=torch.bool, device=qkv.device).triu(1)
    scores = (q @ k.transpose(-1, -2).contiguous() / 8).masked_fill(mask, -math.inf)
    return (torch.softmax(scores, -1) @ v).transpose(1, 2).reshape(b, t, h * 64), torch.logsumexp(scores, -1)


def exact_attention(case, seed, given):
    out, lse, dqkv = [], [], []
    for qkv, grad in zip(given["qkv"], given["grad"]):  # a sequence at a time
        qkv = qkv[None].double().requires_grad_()
        o, s = attend(qkv)
        dqkv.append(torch.autograd.grad(o, qkv, grad[None].double())[0])
        out.append(o.detach())
        lse.append(s.detach())
    return {"out": torch.cat(out), "lse": torch.cat(lse), "dqkv": torch.cat(dqkv)}


def gpt_forward(p, tokens, layers, heads, last_only=False):
    """Logits of kael's GPT (pre-norm blocks, tanh GELU, the head tied to the token table)."""
    functional = torch.nn.functional
    batch, length = tokens.shape
    d = heads * 64

    def norm(x, name):
        return functional.layer_norm(x, (d,), p[name + ".weight"], p[name + ".bias"], EPS)

    def linear(x, name):
        return functional.linear(x, p[name + ".weight"], p[name + ".bias"])

    x = p["token_embedding.weight"][tokens] + p["position_embedding.weight"][:length]
    for layer in range(layers):
        b = f"blocks.{layer}."
        qkv = linear(norm(x, b + "ln1"), b + "attn.qkv").view(batch, length, 3, heads, 64)
        x = x + linear(attend(qkv)[0], b + "attn.proj")
        h = functional.gelu(linear(norm(x, b + "ln2"), b + "mlp.fc1"), approximate="tanh")
        x = x + linear(h, b + "mlp.fc2")
    if last_only:
        x = x[:, -1:]
    return norm(x, "ln_final") @ p["token_embedding.weight"].t()


def exact_gpt_step(case, seed, given):
    p = {n: w.double().requires_grad_() for n, w in given["weights"].items()}
    logits = gpt_forward(p, given["tokens"], case["layers"], case["heads"])
    loss = torch.nn.functional.cross_entropy(logits.flatten(0, 1), given["targets"].flatten())
    grads = dict(zip(p, torch.autograd.grad(loss, list(p.values()))))
    first, second = adam_moments(given["weights"], seed)
    flat, updated = flat_views({n: tuple(w.shape) for n, w in p.items()})
    flat = flat.double()
    _, places = flat_views({n: tuple(w.shape) for n, w in p.items()})
    b1, b2, step = ADAM["beta1"], ADAM["beta2"], ADAM["step"]
    for n in p:
        m = b1 * first[n].double() + (1 - b1) * grads[n]
        v = b2 * second[n].double() + (1 - b2) * grads[n] ** 2
        new = p[n] - ADAM["lr"] * (m / (1 - b1 ** step)) / ((v / (1 - b2 ** step)).sqrt() + ADAM["eps"])
        at = places[n].storage_offset()
        flat[at:at + new.numel()] = new.detach().reshape(-1)
    return {"loss": loss.detach().reshape(1), "grads": grads, "updated": flat}


def exact_prefill(case, seed, given):
    with torch.no_grad():
        p = {n: w.double() for n, w in given["weights"].items()}
        return {"logits": gpt_forward(p, given["prompt"][None], GPT2["layers"], GPT2["heads"], True).reshape(-1)}


def exact_decode(case, seed, given):
    with torch.no_grad():
        p = {n: w.double() for n, w in given["weights"].items()}
        tokens = given["prompt"]
        for i in range(case["tokens"]):
            logits = gpt_forward(p, tokens[None], GPT2["layers"], GPT2["heads"], True).reshape(-1)
            if not case["temperature"]:
                pick = logits.argmax().reshape(1)
            else:
                scaled = logits / case["temperature"]
                if case["top_k"]:
                    scaled = scaled.masked_fill(scaled < scaled.topk(case["top_k"]).values[-1], -math.inf)
                sums = torch.softmax(scaled, 0).cumsum(0)
                pick = (sums > given["uniforms"][i] * sums[-1]).int().argmax().reshape(1)
            tokens = torch.cat([tokens, pick])
        return {"tokens": None, "logits": logits}


def exact_tensor_ops(case, seed, given):
    a, b, c = (given[n].double() for n in ("a", "b", "c"))
    return {"sum": a + b[:, None], "product": a * b[:, None], "transposed": a.t() + c, "scan": a.cumsum(1),
            "row_sum": a.sum(1), "column_sum": a.sum(0), "row_argmax": None, "largest": a.max().reshape(1)}


def exact_rows(case, seed, given):
    x, weight, bias = (given[n].double().requires_grad_() for n in ("x", "weight", "bias"))
    grad = given["grad"].double()
    functional = torch.nn.functional
    y = torch.softmax(x, 1)
    out = {"softmax": y.detach(), "softmax_dx": torch.autograd.grad(y, x, grad)[0]}
    y = functional.layer_norm(x, (case["columns"],), weight, bias, EPS)
    out["norm"] = y.detach()
    out["norm_dx"], out["norm_dweight"], out["norm_dbias"] = torch.autograd.grad(y, (x, weight, bias), grad)
    out["standardized"] = functional.layer_norm(x.detach(), (case["columns"],), None, None, EPS)
    y = functional.gelu(x, approximate="tanh")
    out["gelu"], out["gelu_dx"] = y.detach(), torch.autograd.grad(y, x, grad)[0]
    return out


def mt19937_64(seed, count):
    """The first `count` words of std::mt19937_64(seed), as the C++ standard defines the engine."""
    wrap = (1 << 64) - 1
    words = [seed & wrap]
    for i in range(1, 312):
        words.append((6364136223846793005 * (words[-1] ^ (words[-1] >> 62)) + i) & wrap)
    x = np.array(words, np.uint64)
    upper, lower = np.uint64(wrap ^ 0x7FFFFFFF), np.uint64(0x7FFFFFFF)
    one, matrix = np.uint64(1), np.uint64(0xB5026F5AA96619E9)

    def mixed(high, low, far):
        y = (high & upper) | (low & lower)
        return far ^ (y >> one) ^ np.where(y & one, matrix, np.uint64(0))

    blocks = []
    for _ in range(-(-count // 312)):
        new = np.empty_like(x)
        new[:156] = mixed(x[:156], x[1:157], x[156:])
        new[156:311] = mixed(x[156:311], x[157:], new[:155])
        new[311] = mixed(x[311], new[0], new[155])
        x = new
        blocks.append(x)
    z = np.concatenate(blocks)[:count]
    z = z ^ ((z >> np.uint64(29)) & np.uint64(0x5555555555555555))
    z = z ^ ((z << np.uint64(17)) & np.uint64(0x71D67FFFEDA60000))
    z = z ^ ((z << np.uint64(37)) & np.uint64(0xFFF7EEE000000000))
    return z ^ (z >> np.uint64(43))


def exact_dropout(case, seed, given):
    words = mt19937_64(seed, case["count"])
    mask = torch.from_numpy((words.astype(np.float64) / 2.0 ** 64 < case["keep"]).astype(np.float64)).cuda()
    return {"out": given["x"].double() * mask / case["keep"], "mask": mask, "generator": None}
