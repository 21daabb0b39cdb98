"""The work that programs have this framework's hip device do, case by case, through the tensor API of
vectorcore_amd: whole train steps, prediction, and the single layers and blocks that models are composed of
(a batched product, an activation chain, the loss head, softmax, pooling, feature standardisation), each
with its gradient.

A case is a dict of plain values; `prepare` makes what a program holds before the call, `run` makes one pass,
`exact` is the same pass in 64 bits by plain torch. Results stay on the device, as they do in a program that
goes on computing with them: `run` returns them as Results, a dict that copies an entry to host memory when it
is read. Every device computation of a pass is enqueued within `run`.
"""

import math

import torch

import vectorcore_amd as vc


class Results(dict):
    """Results by name. A device tensor is copied to host memory (a NumPy array) when its entry is read."""

    def __getitem__(self, name):
        value = dict.__getitem__(self, name)
        return value.numpy() if isinstance(value, vc.Tensor) else value


def listed():
    return [
        # A train step of a two-feature, three-class classifier: the smallest, all launches and host work.
        {"name": "spiral_step", "kind": "step", "loss": "xent", "batch": 300, "sizes": "2-64-3", "lr": 1.0},
        # A train step of a digit classifier on a usual batch: still bound by latency.
        {"name": "digits_step", "kind": "step", "loss": "xent", "batch": 256, "sizes": "784-256-10", "lr": 0.1},
        # A train step of a regression whose sizes fit no tile and no 16-byte row.
        {"name": "regression_step", "kind": "step", "loss": "mse", "batch": 999, "sizes": "131-515-515-33", "lr": 0.01},
        # The large train step of the benchmark: bound by matrix products.
        {"name": "mlp_step", "kind": "step", "loss": "xent", "batch": 8192, "sizes": "1024-4096-4096-1000", "lr": 0.01},
        # Class probabilities for one example from the large model: every weight is read for one row.
        {"name": "predict_one", "kind": "predict", "batch": 1, "sizes": "1024-4096-4096-1000"},
        # A batched product with both gradients.
        {"name": "batched_product", "kind": "bmm", "batch": 8, "m": 1024, "k": 1024, "n": 1024, "shared": False},
        # The same on odd sizes, the right operand shared by the batch (its gradient is summed over it).
        {"name": "shared_product_odd", "kind": "bmm", "batch": 48, "m": 197, "k": 65, "n": 131, "shared": True},
        # Bias, two activations and a product of them on a large feature map, with gradients.
        {"name": "activations", "kind": "activations", "rows": 4096, "cols": 4096},
        # The loss head: loss, gradient of the logits, predicted classes.
        {"name": "loss_head", "kind": "loss_head", "rows": 32768, "cols": 1000},
        # Softmax along rows that are not whole 16-byte vectors, with its gradient.
        {"name": "softmax_odd", "kind": "softmax", "rows": 6000, "cols": 1003, "axis": 1, "log": False},
        # Maximum and mean over the middle axis (positions) of [examples, positions, features], with gradient.
        {"name": "pool_positions", "kind": "pool", "outer": 64, "length": 197, "inner": 768, "axis": 1},
        # Each row brought to mean 0 and variance 1, then a gain and an offset per feature, with gradients.
        {"name": "standardise", "kind": "standardise", "rows": 8192, "cols": 1024},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _matrix(rng, rows, cols, most):
    """(rows, cols), each spread over its range's logarithm, of at most `most` elements."""
    while True:
        r, c = _log_int(rng, *rows), _log_int(rng, *cols)
        if r * c <= most:
            return r, c


def draw(rng):
    kind = rng.choice(["step", "predict", "bmm", "activations", "loss_head", "softmax", "pool", "standardise"])
    if kind == "step":
        hidden = [_log_int(rng, 16, 4096) for _ in range(rng.choice([1, 1, 2]))]
        sizes = [_log_int(rng, 2, 1024), *hidden, _log_int(rng, 2, 1000)]
        return {"kind": "step", "loss": rng.choice(["xent", "xent", "mse"]), "batch": _log_int(rng, 16, 8192),
                "sizes": "-".join(map(str, sizes)), "lr": 0.01}
    if kind == "predict":
        hidden = [_log_int(rng, 64, 4096) for _ in range(rng.choice([1, 2]))]
        sizes = [_log_int(rng, 16, 1024), *hidden, _log_int(rng, 2, 1000)]
        return {"kind": "predict", "batch": _log_int(rng, 1, 512), "sizes": "-".join(map(str, sizes))}
    if kind == "bmm":
        while True:
            b, m, k, n = _log_int(rng, 2, 64), *(_log_int(rng, 16, 1024) for _ in range(3))
            if b * m * k * n <= 8 * 1024 ** 3:
                return {"kind": "bmm", "batch": b, "m": m, "k": k, "n": n, "shared": rng.random() < 0.4}
    if kind == "activations":
        rows, cols = _matrix(rng, (32, 16384), (16, 4096), 1 << 24)
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "loss_head":
        rows, cols = _matrix(rng, (32, 32768), (2, 32000), 32768 * 1000)
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "softmax":
        rows, cols = _matrix(rng, (32, 32768), (8, 8192), 1 << 24)
        return {"kind": kind, "rows": rows, "cols": cols, "axis": rng.choice([0, 1, 1, 1]), "log": rng.random() < 0.5}
    if kind == "pool":
        while True:
            o, l, i = _log_int(rng, 2, 512), _log_int(rng, 2, 2048), _log_int(rng, 2, 1024)
            if 4096 <= o * l * i <= 1 << 24:
                return {"kind": kind, "outer": o, "length": l, "inner": i, "axis": rng.choice([0, 1, 1, 2])}
    rows, cols = _matrix(rng, (32, 32768), (16, 4096), 1 << 24)
    return {"kind": "standardise", "rows": rows, "cols": cols}


# ---- inputs ------------------------------------------------------------------


def _sizes(case):
    return [int(s) for s in case["sizes"].split("-")]


def _inputs(case, seed):
    """The pass's inputs by name, as float32 (targets: int64) torch tensors on the GPU, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * scale

    kind = case["kind"]
    if kind in ("step", "predict"):
        dims = _sizes(case)
        v = {"x": normal(case["batch"], dims[0])}
        for i, (fan_in, fan_out) in enumerate(zip(dims[:-1], dims[1:])):
            bound = fan_in ** -0.5
            v["w%d" % i] = (torch.rand(fan_in, fan_out, generator=gen, device="cuda") * 2 - 1) * bound
            v["b%d" % i] = torch.zeros(fan_out, device="cuda") if kind == "step" else normal(fan_out, scale=0.1)
        if kind == "step":
            if case["loss"] == "mse":
                v["targets"] = normal(case["batch"], dims[-1])
            else:
                v["targets"] = torch.randint(dims[-1], (case["batch"],), generator=gen, device="cuda")
        return v
    if kind == "bmm":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return {"a": normal(b, m, k), "b": normal(1 if case["shared"] else b, k, n), "dc": normal(b, m, n)}
    if kind == "pool":
        shape = [case["outer"], case["length"], case["inner"]]
        kept = [s for ax, s in enumerate(shape) if ax != case["axis"]]
        return {"x": normal(*shape), "dy": normal(*kept)}
    rows, cols = case["rows"], case["cols"]
    if kind == "activations":
        return {"x": normal(rows, cols), "bias": normal(1, cols), "dy": normal(rows, cols)}
    if kind == "loss_head":
        return {"logits": normal(rows, cols, scale=2.0),
                "targets": torch.randint(cols, (rows,), generator=gen, device="cuda")}
    if kind == "softmax":
        return {"x": normal(rows, cols, scale=2.0), "dy": normal(rows, cols)}
    return {"x": normal(rows, cols, scale=1.5) + 0.5, "gain": normal(cols, scale=0.1) + 1.0,
            "offset": normal(cols, scale=0.1), "dy": normal(rows, cols)}


# The inputs that a pass differentiates by.
_LEAVES = {"bmm": ("a", "b"), "activations": ("x", "bias"), "loss_head": ("logits",), "softmax": ("x",),
           "pool": ("x",), "standardise": ("x", "gain", "offset")}


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": dict(case)}
    for name, value in _inputs(case, seed).items():
        if value.dtype == torch.int64:
            state[name] = value.cpu().numpy()  # class indices are host data in this API
            continue
        leaf = name in _LEAVES.get(kind, ()) or (kind == "step" and name[0] in "wb")
        state[name] = vc.Tensor(value.cpu().numpy(), requires_grad=leaf, device="hip")
    if kind == "step":
        layers = len(_sizes(case)) - 1
        state["params"] = [state[p + str(i)] for i in range(layers) for p in "wb"]
    vc.synchronize()  # the uploads are done: a program's training loop starts later
    return state


# ---- one pass ----------------------------------------------------------------


def _forward(state, layers):
    h = state["x"]
    for i in range(layers):
        h = h @ state["w%d" % i] + state["b%d" % i]
        if i < layers - 1:
            h = h.relu()
    return h


def _step(state):
    case, params = state["case"], state["params"]
    out = _forward(state, len(params) // 2)
    loss = vc.cross_entropy(out, state["targets"]) if case["loss"] == "xent" else vc.mse_loss(out, state["targets"])
    loss.backward()
    vc.sgd_step(params, case["lr"])
    result = Results(("dw%d" % i, w.grad) for i, w in enumerate(params[::2]))
    vc.zero_grad(params)
    result.update(("p%d" % i, p) for i, p in enumerate(params))
    result["loss"] = loss.item()  # a training loop reads its loss
    return result


def _predict(state):
    logits = _forward(state, len(_sizes(state["case"])) - 1)
    return Results(probabilities=logits.softmax(1), logits=logits)


def _block(state):
    """A block's outputs, and the gradients of its leaves."""
    case = state["case"]
    kind = case["kind"]
    result = Results()
    if kind == "bmm":
        y = result["y"] = state["a"] @ state["b"]
    elif kind == "activations":
        x = state["x"]
        y = result["y"] = (x + state["bias"]).relu().sigmoid() * (x * 0.1).exp()
    elif kind == "softmax":
        x = state["x"]
        y = result["y"] = x.log_softmax(case["axis"]) if case["log"] else x.softmax(case["axis"])
    elif kind == "pool":
        x = state["x"]
        y = result["y"] = x.max(case["axis"]) + x.mean(case["axis"])
        result["where"] = x.argmax(case["axis"])
    else:
        x = state["x"]
        centred = x - x.mean(1, True)
        deviation = (((centred * centred).mean(1, True) + 1e-5).log() * 0.5).exp()
        y = result["y"] = centred / deviation * state["gain"] + state["offset"]
    y.backward(state["dc" if kind == "bmm" else "dy"])
    leaves = _LEAVES[kind]
    result.update(("d" + name, state[name].grad) for name in leaves)
    vc.zero_grad([state[name] for name in leaves])
    return result


def _loss_head(state):
    logits = state["logits"]
    loss = vc.cross_entropy(logits, state["targets"])
    loss.backward()
    result = Results(classes=logits.argmax(1), dlogits=logits.grad, loss=loss.item())
    vc.zero_grad([logits])
    return result


def run(state):
    kind = state["case"]["kind"]
    return {"step": _step, "predict": _predict, "loss_head": _loss_head}.get(kind, _block)(state)


# ---- what a pass cannot do without ---------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("step", "predict"):
        dims, batch = _sizes(case), case["batch"]
        weights = sum(i * o for i, o in zip(dims[:-1], dims[1:]))
        params = weights + sum(dims[1:])
        if kind == "predict":
            return {"bytes": 4 * (batch * (dims[0] + 2 * dims[-1]) + params), "flops": 2 * batch * weights}
        # Forward and weight gradients for every layer, input gradients for all but the first.
        flops = 2 * batch * (3 * weights - dims[0] * dims[1])
        targets = batch * (dims[-1] if case["loss"] == "mse" else 1)
        # Parameters are read and written, their gradients written.
        return {"bytes": 4 * (batch * dims[0] + targets + 3 * params), "flops": flops}
    if kind == "bmm":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        right = (1 if case["shared"] else b) * k * n
        return {"bytes": 4 * 2 * (b * m * k + right + b * m * n), "flops": 6 * b * m * k * n}
    if kind == "pool":
        shape = [case["outer"], case["length"], case["inner"]]
        elements = math.prod(shape)
        kept = elements // shape[case["axis"]]
        return {"bytes": 4 * (2 * elements + 3 * kept), "flops": 3 * elements}
    rows, cols = case["rows"], case["cols"]
    elements = rows * cols
    if kind == "loss_head":
        return {"bytes": 4 * (2 * elements + 2 * rows), "flops": 6 * elements}
    extra = {"activations": 2 * cols, "softmax": 0, "standardise": 4 * cols}[kind]
    # Input and upstream gradient read, result and gradient written.
    return {"bytes": 4 * (4 * elements + extra), "flops": {"activations": 12, "softmax": 8, "standardise": 16}[kind] * elements}


# About four times the largest relative error that each kind shows against `exact` (32-bit sums and products
# throughout; row and column sums are accumulated in double and rounded once).
_TOLERANCE = {"predict": 2e-6, "bmm": 3e-6, "activations": 5e-7, "loss_head": 5e-7, "softmax": 1e-6, "pool": 2e-7,
              "standardise": 5e-7}


def tolerance(case):
    if case["kind"] == "step":
        # A pre-activation within a rounding of 0 falls on either side of the ReLU, and with it one element's
        # whole gradient: about 4e-7 of them do, which is 9e-4 of the gradients' norm for the large step.
        return {"rel": 4e-3, "max": 0.25}
    return {"rel": _TOLERANCE[case["kind"]]}


# ---- the same pass in 64 bits ----------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    v = {k: t if t.dtype == torch.int64 else t.double() for k, t in _inputs(case, seed).items()}
    if kind in ("step", "predict"):
        layers = len(_sizes(case)) - 1
        params = [v[p + str(i)].requires_grad_(kind == "step") for i in range(layers) for p in "wb"]
        h = v["x"]
        for i in range(layers):
            h = h @ params[2 * i] + params[2 * i + 1]
            if i < layers - 1:
                h = h.relu()
        if kind == "predict":
            return {"probabilities": h.softmax(1), "logits": h}
        if case["loss"] == "xent":
            loss = torch.nn.functional.cross_entropy(h, v["targets"])
        else:
            loss = (h - v["targets"]).square().mean()
        grads = torch.autograd.grad(loss, params)
        result = {"dw%d" % i: g for i, g in enumerate(grads[::2])}
        result.update(("p%d" % i, p.detach() - case["lr"] * g) for i, (p, g) in enumerate(zip(params, grads)))
        result["loss"] = float(loss.detach())
        return result
    leaves = _LEAVES[kind]
    for name in leaves:
        v[name].requires_grad_(True)
    result = {}
    if kind == "loss_head":
        loss = torch.nn.functional.cross_entropy(v["logits"], v["targets"])
        grad, = torch.autograd.grad(loss, [v["logits"]])
        classes = v["logits"].detach().argmax(1).double()  # indices come as floats in this API
        return {"classes": classes, "dlogits": grad, "loss": float(loss.detach())}
    if kind == "bmm":
        y = v["a"] @ v["b"].expand(case["batch"], -1, -1)
    elif kind == "activations":
        y = (v["x"] + v["bias"]).relu().sigmoid() * (v["x"] * 0.1).exp()
    elif kind == "softmax":
        y = v["x"].log_softmax(case["axis"]) if case["log"] else v["x"].softmax(case["axis"])
    elif kind == "pool":
        best = v["x"].max(case["axis"])
        y = best.values + v["x"].mean(case["axis"])
        result["where"] = best.indices.double()
    else:
        centred = v["x"] - v["x"].mean(1, keepdim=True)
        y = centred / (centred.square().mean(1, keepdim=True) + 1e-5).sqrt() * v["gain"] + v["offset"]
    grads = torch.autograd.grad(y, [v[name] for name in leaves], v["dc" if kind == "bmm" else "dy"])
    result["y"] = y.detach()
    result.update(("d" + name, g) for name, g in zip(leaves, grads))
    return result
