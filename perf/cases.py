"""Performance cases: the work a program hands to this framework, call by call.

Every case goes through the tensor API (spar_amd.spar) the way a training or
inference program does: a forward pass, and where the path has one the
backward pass from loss = sum(y * G), the loss of the repository's own
benchmark.  The kinds are

  affine      y = x * scale + bias with a per-batch scale and a per-channel
              bias (the headline benchmark's broadcasts), forward and backward
  activation  GELU, SiLU, tanh, sigmoid or the gated silu(a) * b of an MLP
  norm        LayerNorm / RMSNorm over contiguous rows, over a transposed view
              and over a sliced view
  softmax     softmax / log-softmax along the last axis (attention scores, with
              a causal mask added or without) or along a channel axis
  loss        cross entropy of logits, plain or in the language-model form
  reduce      the statistics of a [batch, channel, pixel] tensor: channel sums,
              pixel means, the maximum and its channel, the total
  relayout    attention's head split, its transposed form, the merge back, and
              the rotary embedding read from the two halves of each head
  optimizer   gradient norm, gradient scaling and the AdamW step of a
              transformer's parameter list

A case is a dict of plain values.  `listed()` gives the named cases and
`draw(rng)` one more of the same ranges.
"""
import math

import numpy as np
import torch

from spar_amd import spar

_DTYPES = {"float32": torch.float32, "float64": torch.float64}


# ------------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call: a block of [4, 64, 256] forward and backward, where
        # launches and host time count (the size of the smoke test)
        {"name": "affine_small", "kind": "affine", "batch": 4, "rows": 64, "cols": 256,
         "dtype": "float32"},
        # the headline benchmark's broadcasts at its size
        {"name": "affine_large", "kind": "affine", "batch": 32, "rows": 1024, "cols": 4096,
         "dtype": "float32"},
        # the activation of a transformer MLP over 8192 tokens, training
        {"name": "gelu_tokens", "kind": "activation", "function": "gelu", "rows": 8192,
         "cols": 4096, "dtype": "float32", "train": True},
        # a gated MLP over an odd number of tokens and an odd width
        {"name": "gated_odd", "kind": "activation", "function": "swiglu", "rows": 2047,
         "cols": 2731, "dtype": "float32", "train": True},
        # LayerNorm of 16384 tokens of an ordinary width, training
        {"name": "norm_tokens", "kind": "norm", "function": "layer_norm", "layout": "rows",
         "rows": 16384, "cols": 1024, "dtype": "float32", "train": True},
        # the benchmark's LayerNorm over a transposed view
        {"name": "norm_transposed", "kind": "norm", "function": "layer_norm",
         "layout": "transposed", "rows": 4096, "cols": 8192, "dtype": "float32", "train": True},
        # attention scores of 48 heads over 1024 positions under a causal mask
        {"name": "softmax_attention", "kind": "softmax", "function": "softmax", "outer": 48 * 1024,
         "extent": 1024, "inner": 1, "masked": True, "dtype": "float32", "train": True},
        # class scores per pixel: log-softmax along the channel axis
        {"name": "softmax_channels", "kind": "softmax", "function": "log_softmax", "outer": 16,
         "extent": 256, "inner": 3136, "masked": False, "dtype": "float32", "train": True},
        # a language model's loss over an odd vocabulary
        {"name": "loss_vocabulary", "kind": "loss", "language_model": True, "batch": 4,
         "sequence": 512, "classes": 50257, "dtype": "float32"},
        # per-channel and per-pixel statistics of a batch, in double
        {"name": "statistics_double", "kind": "reduce", "batch": 24, "channels": 96,
         "pixels": 3136, "dtype": "float64"},
        # head split, transpose, merge and rotary embedding of 16 sequences
        {"name": "attention_heads", "kind": "relayout", "batch": 16, "sequence": 1024, "heads": 16,
         "width": 64, "dtype": "float32"},
        # one optimizer step over GPT-2 small's parameter list (124,439,808)
        {"name": "optimizer_step", "kind": "optimizer", "layers": 12, "width": 768,
         "vocabulary": 50257, "positions": 1024, "dtype": "float32"},
    ]


def _log(rng, low, high):
    """A whole number of [low, high], spread over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5)))))))


def draw(rng):
    kind = rng.choice(["affine", "activation", "norm", "softmax", "loss", "reduce", "relayout",
                       "optimizer"])
    dtype = "float32" if rng.random() < 0.85 else "float64"
    most = 1 << 26 if dtype == "float32" else 1 << 25  # elements of a drawn tensor
    train = rng.random() < 0.75
    if kind == "affine":
        cols = _log(rng, 16, 4096)
        rows = _log(rng, 1, 1024)
        return {"kind": kind, "batch": _log(rng, 1, max(1, min(32, most // (rows * cols)))),
                "rows": rows, "cols": cols, "dtype": dtype}
    if kind == "activation":
        function = rng.choice(["gelu", "silu", "tanh", "sigmoid", "swiglu"])
        return {"kind": kind, "function": function, "rows": _log(rng, 1, 8192),
                "cols": _log(rng, 8, 4096), "dtype": dtype, "train": train}
    if kind == "norm":
        function, layout = rng.choice([("layer_norm", "rows"), ("rms_norm", "rows"),
                                       ("layer_norm", "rows"), ("rms_norm", "rows"),
                                       ("layer_norm", "transposed"), ("layer_norm", "sliced")])
        cols = _log(rng, 32, 8192)
        return {"kind": kind, "function": function, "layout": layout,
                "rows": _log(rng, 1, min(16384, most // cols)), "cols": cols, "dtype": dtype,
                "train": train}
    if kind == "softmax":
        function = rng.choice(["softmax", "log_softmax"])
        if rng.random() < 0.35:  # a channel axis
            extent = _log(rng, 2, 1024)
            inner = _log(rng, 2, 4096)
            return {"kind": kind, "function": function,
                    "outer": _log(rng, 1, max(1, min(64, most // (extent * inner)))),
                    "extent": extent, "inner": inner, "masked": False, "dtype": dtype,
                    "train": train}
        masked = rng.random() < 0.4
        extent = _log(rng, 8, 2048) if masked else _log(rng, 8, 40000)
        outer = _log(rng, 1, min(49152, most // extent))
        if masked:  # square score matrices
            outer = max(1, min(outer // extent, 64)) * extent
        return {"kind": kind, "function": function, "outer": outer, "extent": extent, "inner": 1,
                "masked": masked, "dtype": dtype, "train": train}
    if kind == "loss":
        classes = _log(rng, 10, 50257)
        sequence = _log(rng, 2, min(1024, most // classes))
        return {"kind": kind, "language_model": rng.random() < 0.6,
                "batch": _log(rng, 1, max(1, min(8, most // (classes * sequence)))),
                "sequence": sequence, "classes": classes, "dtype": dtype}
    if kind == "reduce":
        pixels = _log(rng, 4, 16384)
        channels = _log(rng, 3, 1024)
        return {"kind": kind, "batch": _log(rng, 1, max(1, min(64, most // (channels * pixels)))),
                "channels": channels, "pixels": pixels, "dtype": dtype}
    if kind == "relayout":
        width = 2 * _log(rng, 8, 64)
        heads = _log(rng, 1, 32)
        sequence = _log(rng, 1, 2048)
        return {"kind": kind,
                "batch": _log(rng, 1, max(1, min(16, (most // 4) // (sequence * heads * width)))),
                "sequence": sequence, "heads": heads, "width": width, "dtype": dtype}
    return {"kind": kind, "layers": _log(rng, 1, 12), "width": 4 * _log(rng, 8, 192),
            "vocabulary": _log(rng, 100, 16384), "positions": _log(rng, 16, 1024),
            "dtype": "float32"}


# ------------------------------------------------------------------ inputs

def _parameter_shapes(case):
    """A decoder-only transformer's parameters: embeddings, then per layer two
    norms, the attention's and the MLP's matrices with their biases, then the
    last norm (GPT-2's list)."""
    c = case["width"]
    shapes = [("tokens", (case["vocabulary"], c)), ("positions", (case["positions"], c))]
    for layer in range(case["layers"]):
        for name, shape in (("norm1.weight", (c,)), ("norm1.bias", (c,)),
                            ("qkv.weight", (c, 3 * c)), ("qkv.bias", (3 * c,)),
                            ("proj.weight", (c, c)), ("proj.bias", (c,)),
                            ("norm2.weight", (c,)), ("norm2.bias", (c,)),
                            ("up.weight", (c, 4 * c)), ("up.bias", (4 * c,)),
                            ("down.weight", (4 * c, c)), ("down.bias", (c,))):
            shapes.append(("%d.%s" % (layer, name), shape))
    return shapes + [("norm.weight", (c,)), ("norm.bias", (c,))]


def _norm_storage(case):
    """Shape of the tensor a norm case's view is taken from."""
    rows, cols = case["rows"], case["cols"]
    if case["layout"] == "transposed":
        return (cols, rows)
    if case["layout"] == "sliced":  # rows [1, rows + 1) and columns [8, cols + 8)
        return (rows + 3, cols + 24)
    return (rows, cols)


def _inputs(case, seed):
    """A case's inputs as torch tensors on the GPU, from the seed alone."""
    device = torch.device("cuda")
    dtype = _DTYPES[case["dtype"]]
    generator = torch.Generator(device=device)
    generator.manual_seed(int(seed) * 1000003 + 17)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=generator, device=device, dtype=dtype) * scale

    def uniform(low, high, *shape):
        return torch.rand(shape, generator=generator, device=device, dtype=dtype) * (high - low) + low

    kind = case["kind"]
    if kind == "affine":
        b, r, c = case["batch"], case["rows"], case["cols"]
        return {"x": normal(b, r, c), "scale": uniform(0.5, 1.5, b, 1, c),
                "bias": uniform(-0.1, 0.1, c), "G": normal(b, r, c)}
    if kind == "activation":
        shape = (case["rows"], case["cols"])
        made = {"x": normal(*shape, scale=1.5)}
        if case["function"] == "swiglu":
            made["b"] = normal(*shape)
        if case["train"]:
            made["G"] = normal(*shape)
        return made
    if kind == "norm":
        made = {"x": normal(*_norm_storage(case)) + 0.25,
                "weight": uniform(0.5, 1.5, case["cols"]), "bias": uniform(-0.1, 0.1, case["cols"])}
        if case["train"]:
            made["G"] = normal(case["rows"], case["cols"])
        return made
    if kind == "softmax":
        shape = ((case["outer"], case["extent"]) if case["inner"] == 1
                 else (case["outer"], case["extent"], case["inner"]))
        if case["masked"]:
            n = case["extent"]
            shape = (case["outer"] // n, n, n)
        made = {"x": normal(*shape, scale=2.0)}
        if case["masked"]:
            made["mask"] = torch.triu(torch.full((n, n), -math.inf, device=device, dtype=dtype), 1)
        if case["train"]:
            made["G"] = normal(*shape)
        return made
    if kind == "loss":
        shape = (case["batch"], case["sequence"])
        return {"logits": normal(*shape, case["classes"], scale=2.0),
                "targets": torch.randint(0, case["classes"], shape, generator=generator,
                                         device=device, dtype=torch.int64)}
    if kind == "reduce":
        return {"x": normal(case["batch"], case["channels"], case["pixels"]) + 1.0}
    if kind == "relayout":
        t, d = case["sequence"], case["width"]
        angle = (torch.arange(t, device=device, dtype=torch.float64)[:, None, None]
                 * torch.exp(torch.arange(d // 2, device=device, dtype=torch.float64)
                             * (-math.log(10000.0) / (d // 2))))
        return {"x": normal(case["batch"], t, case["heads"] * d), "cos": torch.cos(angle).to(dtype),
                "sin": torch.sin(angle).to(dtype)}
    shapes = _parameter_shapes(case)
    total = sum(math.prod(shape) for _, shape in shapes)
    return {"values": normal(total, scale=0.02), "gradients": normal(total, scale=0.001)}


# ------------------------------------------------------------- preparation

_CPU = spar.Device.cpu()


def _to_device(array):
    return spar.Tensor.from_numpy(array).to(spar.Device.hip(0))


def prepare(case, seed):
    """What a program holds before the call: its tensors on the device, with
    the trained ones marked, and for the optimizer the parameters with their
    gradients and the optimizer over them."""
    made = _inputs(case, seed)
    state = {"case": case}
    if case["kind"] == "optimizer":
        values, gradients = (made[k].cpu().numpy() for k in ("values", "gradients"))
        parameters, at = [], 0
        for _, shape in _parameter_shapes(case):
            end = at + math.prod(shape)
            parameter = spar.nn.Parameter(_to_device(values[at:end].reshape(shape)))
            gradient = _to_device(gradients[at:end].reshape(shape))
            spar.sum(spar.multiply(parameter.tensor(), gradient)).backward()  # grad = gradient
            parameters.append(parameter)
            at = end
        state["parameters"] = parameters
        state["optimizer"] = spar.optim.AdamW(parameters, learning_rate=1e-3, weight_decay=0.01)
        return state
    trained = {"affine": ("x", "scale", "bias"), "activation": ("x", "b"),
               "norm": ("x", "weight", "bias"), "softmax": ("x",), "loss": ("logits",)}
    for name, value in made.items():
        if name == "bias" and case.get("function") == "rms_norm":
            continue
        tensor = _to_device(value.cpu().numpy())
        if name in trained.get(case["kind"], ()) and case.get("train", True):
            tensor.set_requires_grad(True)
        state[name] = tensor
    return state


# --------------------------------------------------------------- one pass

class Results(dict):
    """A pass's outputs by name.  An entry is copied to host memory when it is
    read, as a program does with the results it looks at, so that the pass
    itself neither copies nor waits."""

    def __getitem__(self, name):
        value = super().__getitem__(name)
        if callable(value):
            value = value()
        if isinstance(value, list):
            return np.concatenate([t.to(_CPU).numpy().reshape(-1) for t in value])
        return value.to(_CPU).numpy() if isinstance(value, spar.Tensor) else value


def _backward(state, results, output, names):
    """Backward of loss = sum(output * G), and the named leaves' gradients.
    (The loss itself carries G to the output; a sum of as many positive as
    negative terms, it has no stable relative error and is not compared.)"""
    return _gradients(state, results, spar.sum(spar.multiply(output, state["G"])), names)


def _gradients(state, results, loss, names):
    for name in names:
        state[name].zero_grad()
    loss.backward()
    for name in names:
        results["d" + name] = state[name].grad()
    return results


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "affine":
        y = spar.add(spar.multiply(state["x"], state["scale"]), state["bias"])
        return _backward(state, Results(y=y), y, ("x", "scale", "bias"))
    if kind == "activation":
        if case["function"] == "swiglu":
            y = spar.multiply(spar.silu(state["x"]), state["b"])
            names = ("x", "b")
        else:
            y = getattr(spar, case["function"])(state["x"])
            names = ("x",)
        results = Results(y=y)
        return _backward(state, results, y, names) if case["train"] else results
    if kind == "norm":
        x = state["x"]
        if case["layout"] == "transposed":
            x = x.transpose(0, 1)
        elif case["layout"] == "sliced":
            x = x.narrow(0, 1, case["rows"]).narrow(1, 8, case["cols"])
        if case["function"] == "layer_norm":
            y = spar.layer_norm(x, state["weight"], state["bias"])
            names = ("x", "weight", "bias")
        else:
            y = spar.rms_norm(x, state["weight"])
            names = ("x", "weight")
        results = Results(y=y)
        return _backward(state, results, y, names) if case["train"] else results
    if kind == "softmax":
        x = state["x"]
        if case["masked"]:
            x = spar.add(x, state["mask"])
        axis = 2 if case["masked"] else 1
        y = getattr(spar, case["function"])(x, axis)
        results = Results(y=y)
        if not case["train"]:
            return results
        if case["function"] == "log_softmax" and case["masked"]:
            # log-probabilities are -inf above the diagonal: a weighted sum of
            # their exponentials is what such a program differentiates
            return _backward(state, results, spar.exp(y), ("x",))
        return _backward(state, results, y, ("x",))
    if kind == "loss":
        if case["language_model"]:
            loss = spar.loss.language_model_cross_entropy(state["logits"], state["targets"])
        else:
            loss = spar.loss.cross_entropy(state["logits"], state["targets"])
        return _gradients(state, Results(loss=loss), loss, ("logits",))
    if kind == "reduce":
        x = state["x"]
        return Results(channel_sum=spar.sum(x, [0, 2]), pixel_mean=spar.mean(x, 2),
                       peak=spar.max(x, 1), which=spar.argmax(x, 1), total=spar.sum(x))
    if kind == "relayout":
        b, t, h, d = case["batch"], case["sequence"], case["heads"], case["width"]
        heads = state["x"].reshape([b, t, h, d])
        split = heads.permute([0, 2, 1, 3]).contiguous()       # queries [b, h, t, d]
        transposed = heads.permute([0, 2, 3, 1]).contiguous()  # keys [b, h, d, t]
        merged = split.permute([0, 2, 1, 3]).contiguous()      # back to [b, t, h, d]
        first, second = heads.narrow(3, 0, d // 2), heads.narrow(3, d // 2, d // 2)
        cos, sin = state["cos"], state["sin"]
        return Results(split=split, transposed=transposed, merged=merged,
                       rotated_first=spar.subtract(spar.multiply(first, cos),
                                                   spar.multiply(second, sin)),
                       rotated_second=spar.add(spar.multiply(second, cos),
                                               spar.multiply(first, sin)))
    # clip_grad_norm's two halves, always both: the gradients of a pass are
    # the last pass's, whose norm a first clip leaves at the limit
    parameters, optimizer = state["parameters"], state["optimizer"]
    norm = spar.training.global_grad_norm(parameters)
    spar.training.scale_gradients(parameters, 1.0 / norm)
    optimizer.step()

    def moment(name):
        return lambda: [getattr(optimizer.parameter_state(p), name) for p in parameters]

    return Results(norm=norm, parameters=lambda: [p.tensor() for p in parameters],
                   gradients=lambda: [p.grad() for p in parameters],
                   first=moment("first_moment"), second=moment("second_moment"))


# ------------------------------------------------------------ measurements

def _elements(case):
    kind = case["kind"]
    if kind == "affine":
        return case["batch"] * case["rows"] * case["cols"]
    if kind in ("activation", "norm"):
        return case["rows"] * case["cols"]
    if kind == "softmax":
        return case["outer"] * case["extent"] * case["inner"]
    if kind == "loss":
        return case["batch"] * case["sequence"] * case["classes"]
    if kind == "reduce":
        return case["batch"] * case["channels"] * case["pixels"]
    if kind == "relayout":
        return case["batch"] * case["sequence"] * case["heads"] * case["width"]
    return sum(math.prod(shape) for _, shape in _parameter_shapes(case))


def work(case):
    """Each input read once, each output written once, and a few operations
    per element."""
    n = _elements(case)
    kind = case["kind"]
    train = case.get("train", True)
    item = 4 if case["dtype"] == "float32" else 8
    if kind == "affine":  # x, G; y, dx; scale, bias and their gradients
        values = 4 * n + 2 * (case["batch"] + 1) * case["cols"]
        flops = 8 * n
    elif kind == "activation":  # x (b), G; y, dx (db)
        pair = case["function"] == "swiglu"
        values = (3 if pair else 2) * n + ((3 if pair else 2) * n if train else 0)
        flops = (40 if train else 20) * n
    elif kind == "norm":  # x, G; y, dx (of the storage the view is taken from)
        values = 2 * n + (n + math.prod(_norm_storage(case)) if train else 0) + 4 * case["cols"]
        flops = (18 if train else 8) * n
    elif kind == "softmax":  # x (mask), G; y, dx
        values = (4 if train else 2) * n + (case["extent"] ** 2 if case["masked"] else 0)
        flops = (14 if train else 8) * n
    elif kind == "loss":  # logits; their gradient
        values = 2 * n + 2 * case["batch"] * case["sequence"]
        flops = 12 * n
    elif kind == "reduce":  # x; the five results (argmax's are 8 bytes each)
        b, c, s = case["batch"], case["channels"], case["pixels"]
        values = n + c + b * c + b * s * (1 + 8 // item) + 1
        flops = 5 * n
    elif kind == "relayout":  # x; four results of its size
        values = 5 * n + case["sequence"] * case["width"]
        flops = 3 * n
    else:  # parameters, gradients and both moments, read and written
        values = 8 * n
        flops = 18 * n
    return {"bytes": values * item, "flops": flops}


def tolerance(case):
    """About four times the largest error against 64 bits over the listed
    cases and 150 drawn ones: in float32 2.5e-7 relative for column sums and
    norms, 4e-7 for the softmax family (whose exponentials and row sums it
    holds), 6e-8 for the optimizer's values; in float64 3.4e-16."""
    if case["dtype"] == "float64":
        return {"rel": 2e-15, "max": 4e-14}
    if case["kind"] == "optimizer":
        return {"rel": 3e-7, "max": 1e-6}
    if case["kind"] in ("softmax", "loss"):
        return {"rel": 2e-6, "max": 5e-5}
    return {"rel": 1e-6, "max": 1e-5}


# ---------------------------------------------------------- 64-bit results

def _norm_view(case, x):
    if case["layout"] == "transposed":
        return x.t()
    if case["layout"] == "sliced":
        return x[1:case["rows"] + 1, 8:case["cols"] + 8]
    return x


def exact(case, seed):
    """run()'s results of the same inputs from plain torch in float64."""
    kind = case["kind"]
    made = _inputs(case, seed)
    if kind == "optimizer":
        p, g = made["values"].double(), made["gradients"].double()
        norm = float(torch.linalg.vector_norm(g))
        g *= 1.0 / norm
        first, second = 0.1 * g, 0.001 * g * g
        p *= 1.0 - 1e-3 * 0.01
        p -= 1e-3 * (first / (1.0 - 0.9)) / ((second / (1.0 - 0.999)).sqrt() + 1e-8)
        return {"norm": norm, "parameters": p, "gradients": g, "first": first, "second": second}
    if kind == "reduce":
        x = made["x"].double()
        return {"channel_sum": x.sum((0, 2)), "pixel_mean": x.mean(2), "peak": x.amax(1),
                "which": None, "total": x.sum()}
    if kind == "relayout":
        b, t, h, d = case["batch"], case["sequence"], case["heads"], case["width"]
        heads = made["x"].double().reshape(b, t, h, d)
        first, second = heads[..., :d // 2], heads[..., d // 2:]
        cos, sin = made["cos"].double(), made["sin"].double()
        return {"split": heads.permute(0, 2, 1, 3).contiguous(),
                "transposed": heads.permute(0, 2, 3, 1).contiguous(), "merged": heads,
                "rotated_first": first * cos - second * sin,
                "rotated_second": second * cos + first * sin}
    if kind == "loss":
        z = made["logits"].double()
        targets = made["targets"]
        if case["language_model"]:
            z_used, targets = z[:, :-1], targets[:, 1:]
        else:
            z_used = z
        log_p = torch.log_softmax(z_used, -1)
        count = targets.numel()
        loss = -log_p.gather(-1, targets[..., None]).sum() / count
        used = log_p.exp_().scatter_add_(-1, targets[..., None],
                                         torch.full(targets.shape + (1,), -1.0, device=z.device,
                                                    dtype=torch.float64)).div_(count)
        if not case["language_model"]:
            return {"loss": loss, "dlogits": used}
        gradient = torch.zeros_like(z)
        gradient[:, :-1] = used
        return {"loss": loss, "dlogits": gradient}

    made = {name: value.double() for name, value in made.items()}
    names = {"affine": ("x", "scale", "bias"), "activation": ("x", "b"),
             "norm": ("x", "weight", "bias"), "softmax": ("x",)}[kind]
    names = [n for n in names if n in made]
    train = case.get("train", True)
    if train:
        for name in names:
            made[name].requires_grad_(True)
    weigh = None
    if kind == "affine":
        y = made["x"] * made["scale"] + made["bias"]
    elif kind == "activation":
        x = made["x"]
        y = {"gelu": torch.nn.functional.gelu, "silu": torch.nn.functional.silu,
             "tanh": torch.tanh, "sigmoid": torch.sigmoid,
             "swiglu": lambda v: torch.nn.functional.silu(v) * made["b"]}[case["function"]](x)
    elif kind == "norm":
        x = _norm_view(case, made["x"])
        if case["function"] == "layer_norm":
            centred = x - x.mean(1, keepdim=True)
            y = (centred / (centred.square().mean(1, keepdim=True) + 1e-5).sqrt() * made["weight"]
                 + made["bias"])
        else:
            names = ["x", "weight"]
            y = x / (x.square().mean(1, keepdim=True) + 1e-5).sqrt() * made["weight"]
    else:
        x = made["x"] + made["mask"] if case["masked"] else made["x"]
        y = getattr(torch, case["function"])(x, 2 if case["masked"] else 1)
        if case["function"] == "log_softmax" and case["masked"]:
            weigh = torch.softmax(x, 2)
    result = {"y": y.detach()}
    if not train:
        return result
    loss = ((y if weigh is None else weigh) * made["G"]).sum()
    gradients = torch.autograd.grad(loss, [made[name] for name in names])
    for name, gradient in zip(names, gradients):
        result["d" + name] = gradient
    return result
