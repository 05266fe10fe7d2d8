"""Workloads of the fused residual + dropout + LayerNorm, as programs call it.

Four ways of calling, each through a public entry point:

* ``call``: one ``residual_layer_norm`` without a graph to record, as a served
  model's prefill and decode steps make it (host cost included).
* ``step``: ``residual_layer_norm`` and ``torch.autograd.grad`` of both
  outputs, the op's part of an eager training step; ``deterministic`` runs it
  under ``torch.use_deterministic_algorithms(True)``, ``frozen`` with
  weight and bias that need no gradient.
* ``buffers``: forward and backward through the C ABI on buffers the caller
  owns (a trainer with its own memory planning, or a captured region).
* ``decode_graph`` / ``train_graph``: every residual norm of a stack of
  ``layers`` captured into one HIP graph, as launch-bound decode loops and
  small training steps run.

A case names its rows as ``batch`` x ``length``; ``offset`` is the mean of x.
``exact`` evaluates the same op in float64 with plain torch operations, the
dropout masks included (Philox4x32-10, Salmon et al., SC'11, in the layouts
that include/rln.h defines).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGES = str(Path(__file__).resolve().parent.parent / "gfx1010-kernels_amd")
if _PACKAGES not in sys.path:
    sys.path.insert(0, _PACKAGES)

EPS = 1e-5
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
SIZES = {"float32": 4, "float16": 2, "bfloat16": 2}
# Hidden sizes with kernels of their own, and the dropout launch width that
# names their mask layout; every other multiple of 64 uses the library's.
WIDTHS = {128: 128, 256: 128, 384: 128, 512: 128, 768: 128, 1024: 192}


def _case(name, kind, batch, length, hidden, branch, normalized="float32", p=0.0,
          deterministic=False, frozen=False, layers=1, offset=0.0):
    case = dict(kind=kind, batch=batch, length=length, hidden=hidden, branch=branch,
                normalized=normalized, p=p, deterministic=deterministic, frozen=frozen,
                layers=layers, offset=offset)
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # A decode step of a served GPT-2-small-shaped model: one token for each
        # of 8 sequences, bf16 activations, one eager call under no_grad.
        _case("decode_call", "call", 8, 1, 768, "bfloat16", "bfloat16"),
        # The 24 residual norms of one decode step of a 12-block stack, 64
        # sequences, hidden 1600, in one HIP graph.
        _case("decode_stack", "decode_graph", 64, 1, 1600, "float16", "float16", layers=24),
        # Evaluation of a [4, 1024, 768] batch in fp32 (forward only).
        _case("eval_batch", "call", 4, 1024, 768, "float32"),
        # Prefill of one ragged long prompt in bf16, a hidden size that is
        # served by the kernels with a run-time row length.
        _case("prefill_ragged", "call", 1, 6001, 2880, "bfloat16", "bfloat16"),
        # The character-level GPT's training microstep, B = 1, T = 1024, C =
        # 384: an eager step of one norm ...
        _case("char_gpt_norm", "step", 1, 1024, 384, "float16", p=0.15),
        # ... and 12 residual norms (six blocks), forward and backward, captured.
        _case("char_gpt_stack", "train_graph", 1, 1024, 384, "float16", p=0.15, layers=12),
        # GPT-2-small-shaped training batch, the benchmark's default workload.
        _case("train_768", "buffers", 8, 1024, 768, "float16", p=0.1),
        # fp32 branch, an odd row count and a residual stream far from zero mean.
        _case("train_tail", "buffers", 3, 4097, 384, "float32", p=0.1, offset=100.0),
        # The same batch at hidden 1600 (two to four waves per row).
        _case("train_1600", "buffers", 8, 1024, 1600, "bfloat16", p=0.1),
        # Deterministic training, fixed-order weight and bias gradients.
        _case("deterministic", "step", 32, 2048, 1024, "float16", p=0.15, deterministic=True),
        # Large training batches: the smallest hidden size in fp16, ...
        _case("train_large_128", "step", 64, 4096, 128, "float16", p=0.15),
        # ... and hidden 768 with bf16 in, bf16 out.
        _case("train_large_768", "step", 64, 4096, 768, "bfloat16", "bfloat16", p=0.15),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    """One more case: any kind, hidden size, dtypes and option, with sizes
    spread over the logarithm of each kind's range and ragged row counts."""
    kind = rng.choice(["call", "step", "step", "buffers", "decode_graph", "train_graph"])
    if rng.random() < 0.5:
        hidden = rng.choice(sorted(WIDTHS))
    else:
        hidden = 64 * round(_log_uniform(rng, 2, 128))
    # Elements of one tensor: a token to a large batch; a graph's stack is small.
    low, high = {"call": (hidden, 1 << 26), "step": (1 << 16, 1 << 27),
                 "buffers": (1 << 18, 1 << 25), "decode_graph": (hidden, 1 << 19),
                 "train_graph": (1 << 17, 1 << 22)}[kind]
    rows = max(1, round(_log_uniform(rng, max(low, hidden), max(high, 2 * hidden)) / hidden))
    batch = min(rows, rng.choice([1, 1, 2, 3, 8]))
    branch = rng.choice(["float16", "bfloat16", "float32"])
    normalized = rng.choice(["float32", branch])
    training = kind in ("step", "buffers", "train_graph")
    return _case(
        None, kind, batch, max(1, rows // batch), hidden, branch, normalized,
        p=rng.choice([0.0, 0.1, 0.15, round(rng.uniform(0.05, 0.5), 3)]) if training else 0.0,
        deterministic=kind in ("step", "buffers") and rng.random() < 0.25,
        frozen=kind == "step" and rng.random() < 0.2,
        layers={"decode_graph": rng.choice([8, 12, 24]),
                "train_graph": rng.choice([4, 8, 12])}.get(kind, 1),
        offset=rng.choice([0.0, 0.0, 0.0, round(rng.uniform(-20, 20), 2)]))


def _inputs(case, seed):
    """Inputs of every layer, from the seed alone: x, and per layer a branch,
    weight, bias and upstream gradients (of `normalized`; and of the last
    `updated`)."""
    generator = torch.Generator("cuda").manual_seed(seed)
    shape = (case["batch"], case["length"], case["hidden"])

    def normal(size, scale=1.0, mean=0.0, dtype=torch.float32):
        values = torch.randn(size, device="cuda", generator=generator)
        return values.mul_(scale).add_(mean).to(dtype)

    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(
            branch=normal(shape, 0.5, dtype=DTYPES[case["branch"]]),
            weight=normal(case["hidden"], 0.02, 1.0),
            bias=normal(case["hidden"], 0.02)))
    x = normal(shape, mean=case["offset"])
    grad_updated = None
    if case["kind"] in ("step", "buffers", "train_graph"):
        grad_updated = normal(shape)
        for layer in layers:
            layer["grad_normalized"] = normal(shape, dtype=DTYPES[case["normalized"]])
    return x, layers, grad_updated


def _train_stack(state):
    """Forward through every layer, then the gradients of all inputs."""
    from gfx1010_kernels import residual_layer_norm

    x = state["x"]
    normalized, inputs = [], [x]
    for layer in state["layers"]:
        x, y = residual_layer_norm(x, layer["branch"], layer["weight"], layer["bias"],
                                   state["p"], EPS, True, normalized_dtype=state["dtype"])
        normalized.append(y)
        inputs.append(layer["branch"])
        if not state["frozen"]:
            inputs += [layer["weight"], layer["bias"]]
    gradients = torch.autograd.grad(
        [x, *normalized], inputs,
        [state["grad_updated"], *(layer["grad_normalized"] for layer in state["layers"])])
    return [x, *normalized, *gradients]


def _decode_stack(state):
    from gfx1010_kernels import residual_layer_norm

    x, outputs = state["x"], []
    with torch.no_grad():
        for layer in state["layers"]:
            x, y = residual_layer_norm(x, layer["branch"], layer["weight"], layer["bias"],
                                       0.0, EPS, False, normalized_dtype=state["dtype"])
            outputs.append(y)
    return [x, *outputs]


def _buffers(case, state):
    """Output buffers and argument lists of the C ABI calls, built once."""
    from gfx1010_kernels import _cabi

    codes = {"float32": _cabi.RLN_DTYPE_F32, "float16": _cabi.RLN_DTYPE_F16,
             "bfloat16": _cabi.RLN_DTYPE_BF16}
    x, layer = state["x"], state["layers"][0]
    hidden = case["hidden"]
    rows = case["batch"] * case["length"]
    dropout = case["p"] > 0.0
    words = rows * hidden // 32 if dropout else 0
    out = {
        "updated": torch.empty_like(x),
        "normalized": torch.empty_like(x, dtype=state["dtype"]),
        "mean": torch.empty(rows, device="cuda"),
        "rstd": torch.empty(rows, device="cuda"),
        "mask": torch.empty(words, dtype=torch.int32, device="cuda"),
        "grad_x": torch.empty_like(x),
        "grad_branch": torch.empty_like(layer["branch"]),
        "grad_weight": torch.empty(hidden, device="cuda"),
        "grad_bias": torch.empty(hidden, device="cuda"),
    }
    at = {name: tensor.data_ptr() if tensor.numel() else None for name, tensor in out.items()}
    workspace_bytes = _cabi.backward_workspace_bytes(rows, hidden, case["deterministic"])
    workspace = torch.empty(workspace_bytes, dtype=torch.uint8, device="cuda")
    philox = None
    if dropout:
        philox = _cabi.RlnPhilox(seed=state["seed"], offset=0, seed_ptr=None, offset_ptr=None,
                                 threads=WIDTHS.get(hidden, 0))
    weight, bias = layer["weight"].data_ptr(), layer["bias"].data_ptr()
    forward = dict(
        x=x.data_ptr(), branch=layer["branch"].data_ptr(), branch_dtype=codes[case["branch"]],
        weight=weight, bias=bias, updated=at["updated"], normalized=at["normalized"],
        mean=at["mean"], rstd=at["rstd"], mask=at["mask"], rows=rows, hidden=hidden,
        dropout_p=case["p"], eps=EPS, training=True, philox=philox,
        normalized_dtype=codes[case["normalized"]], zero_grad_weight=at["grad_weight"],
        zero_grad_bias=at["grad_bias"])
    backward = dict(
        grad_updated=state["grad_updated"].data_ptr(),
        grad_normalized=layer["grad_normalized"].data_ptr(), updated=at["updated"],
        weight=weight, mean=at["mean"], rstd=at["rstd"], mask=at["mask"], grad_x=at["grad_x"],
        grad_branch=at["grad_branch"], branch_dtype=codes[case["branch"]],
        grad_weight=at["grad_weight"], grad_bias=at["grad_bias"], rows=rows, hidden=hidden,
        dropout_p=case["p"], training=True, deterministic=case["deterministic"],
        workspace=workspace.data_ptr() if workspace_bytes else None,
        workspace_bytes=workspace_bytes, accumulate_parameters=True,
        grad_normalized_dtype=codes[case["normalized"]])
    state.update(out=out, workspace=workspace, forward=forward, backward=backward)


def prepare(case, seed):
    # Once per program, as a trainer sets it.
    torch.use_deterministic_algorithms(case["deterministic"])
    x, layers, grad_updated = _inputs(case, seed)
    kind = case["kind"]
    state = dict(kind=kind, x=x, layers=layers, grad_updated=grad_updated, p=case["p"],
                 dtype=DTYPES[case["normalized"]], frozen=case["frozen"], seed=seed)
    if kind in ("step", "train_graph"):
        x.requires_grad_()
        for layer in layers:
            layer["branch"].requires_grad_()
            if not case["frozen"]:
                layer["weight"].requires_grad_()
                layer["bias"].requires_grad_()
    elif kind == "buffers":
        _buffers(case, state)
    if kind.endswith("graph"):
        stack = _decode_stack if kind == "decode_graph" else _train_stack
        graph = torch.cuda.CUDAGraph()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            stack(state)  # the first call outside the capture, as capture wants it
        torch.cuda.current_stream().wait_stream(side)
        with torch.cuda.graph(graph):
            outputs = stack(state)
        state.update(graph=graph, outputs=outputs)
    torch.cuda.manual_seed(seed)
    return state


def run(state):
    kind = state["kind"]
    if kind == "call":
        from gfx1010_kernels import residual_layer_norm

        layer = state["layers"][0]
        with torch.no_grad():
            return residual_layer_norm(state["x"], layer["branch"], layer["weight"],
                                       layer["bias"], 0.0, EPS, False,
                                       normalized_dtype=state["dtype"])
    if kind == "step":
        return _train_stack(state)
    if kind == "buffers":
        from gfx1010_kernels import _cabi

        stream = torch.cuda.current_stream().cuda_stream
        _cabi.forward(stream=stream, **state["forward"])
        _cabi.backward(stream=stream, **state["backward"])
        return state["out"]
    state["graph"].replay()
    return state["outputs"]


def work(case):
    """Compulsory traffic: every input read once, every output written once,
    what a training forward keeps for its backward written and read once."""
    rows = case["batch"] * case["length"]
    hidden = case["hidden"]
    branch, normalized = SIZES[case["branch"]], SIZES[case["normalized"]]
    count = rows * hidden
    total = count * (4 + branch + 4 + normalized) + 8 * hidden  # x, branch -> updated, normalized
    flops = 10.0 * count
    if case["kind"] in ("step", "buffers", "train_graph"):
        # updated and both upstream gradients -> grad_x, grad_branch
        total += count * (4 + 4 + normalized + 4 + branch) + 4 * hidden
        total += 2 * 8 * rows  # mean and rstd
        if case["p"] > 0.0:
            total += 2 * (count // 8)  # the mask
        if not case["frozen"]:
            total += 8 * hidden
        flops += 20.0 * count
    return {"bytes": case["layers"] * total, "flops": case["layers"] * flops}


def tolerance(case):
    """fp32 outputs: a float64 evaluation is 5e-6 away where the mean of x is
    100 times its spread (the rounding of x + branch), 1e-7 elsewhere.
    16-bit outputs: 2.1e-4 (fp16) and 1.7e-3 (bf16) away, their rounding.
    Four times that, and two ulps of the output type at most."""
    kinds = {case["branch"] if case["kind"] in ("step", "buffers", "train_graph") else "float32",
             case["normalized"]}
    if "bfloat16" in kinds:
        return {"rel": 7e-3, "max": 1.6e-2}
    if "float16" in kinds:
        return {"rel": 8.5e-4, "max": 2e-3}
    return {"rel": 2e-5, "max": 4e-4}


def _philox(counter, seed):
    """Philox4x32-10 of the four counter words (int64 tensors of 32-bit values)."""
    low = 0xFFFFFFFF
    c0, c1, c2, c3 = counter
    k0, k1 = seed & low, (seed >> 32) & low
    for _ in range(10):
        product0, product1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((product1 >> 32) & low) ^ c1 ^ k0, product1 & low,
                          ((product0 >> 32) & low) ^ c3 ^ k1, product0 & low)
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c0, c1, c2, c3


def _increment(hidden):
    threads = WIDTHS.get(hidden, 0)
    return 4 if threads == 0 else 4 * -(-(-(-hidden // threads)) // 4)


def _keep(first, rows, hidden, seed, offset, p):
    """Keep flags of rows first .. first + rows - 1 for a draw at `offset`."""
    threshold = int(float(torch.tensor(p, dtype=torch.float32)) * 4294967296.0)
    row = torch.arange(first, first + rows, device="cuda", dtype=torch.int64)[:, None]
    threads = WIDTHS.get(hidden, 0)
    if threads == 0:
        group = row * (hidden // 4) + torch.arange(hidden // 4, device="cuda")
        words = _philox((torch.full_like(group, offset // 4), torch.zeros_like(group),
                         group & 0xFFFFFFFF, group >> 32), seed)
        return torch.stack(words, -1).reshape(rows, hidden) >= threshold
    stream = row * threads + torch.arange(threads, device="cuda")
    items = []
    for call in range(_increment(hidden) // 4):
        items += _philox((torch.full_like(stream, offset // 4 + call), torch.zeros_like(stream),
                          stream & 0xFFFFFFFF, stream >> 32), seed)
    return torch.cat(items, -1)[:, :hidden] >= threshold


def _chunks(rows, hidden):
    step = max(1, (1 << 23) // hidden)
    return [(first, min(rows, first + step)) for first in range(0, rows, step)]


def exact(case, seed):
    x, layers, grad_updated = _inputs(case, seed)
    hidden, p = case["hidden"], case["p"]
    rows = case["batch"] * case["length"]
    training = grad_updated is not None
    dropout = training and p > 0.0
    scale = float(torch.tensor(1.0) / (torch.tensor(1.0) - torch.tensor(p)))
    double = dict(dtype=torch.float64, device="cuda")
    current = x.view(rows, hidden)
    forward = []
    for index, layer in enumerate(layers):
        out = dict(updated=torch.empty(rows, hidden, **double),
                   normalized=torch.empty(rows, hidden, **double),
                   mean=torch.empty(rows, **double), rstd=torch.empty(rows, **double))
        weight, bias = layer["weight"].double(), layer["bias"].double()
        branch = layer["branch"].view(rows, hidden)
        for a, b in _chunks(rows, hidden):
            dropped = branch[a:b]
            if dropout:
                # The dropped branch is rounded to the branch's type, once.
                keep = _keep(a, b - a, hidden, seed, index * _increment(hidden), p)
                dropped = (dropped.float() * keep * scale).to(dropped.dtype)
            u = current[a:b].double() + dropped.double()
            mean = u.mean(-1, keepdim=True)
            rstd = (u.var(-1, unbiased=False, keepdim=True) + EPS).rsqrt()
            out["updated"][a:b] = u
            out["normalized"][a:b] = (u - mean) * rstd * weight + bias
            out["mean"][a:b] = mean[:, 0]
            out["rstd"][a:b] = rstd[:, 0]
        forward.append(out)
        current = out["updated"]
    if not training:
        return [current, *(out["normalized"] for out in forward)]
    upstream = grad_updated.view(rows, hidden)
    gradients = []
    for index in reversed(range(len(layers))):
        layer, out = layers[index], forward[index]
        grad_x = torch.empty(rows, hidden, **double)
        grad_branch = torch.empty(rows, hidden, **double)
        grad_weight, grad_bias = torch.zeros(hidden, **double), torch.zeros(hidden, **double)
        grad_normalized = layer["grad_normalized"].view(rows, hidden)
        weight = layer["weight"].double()
        for a, b in _chunks(rows, hidden):
            gy = grad_normalized[a:b].double()
            rstd = out["rstd"][a:b, None]
            xhat = (out["updated"][a:b] - out["mean"][a:b, None]) * rstd
            q = gy * weight
            g = upstream[a:b].double() + rstd * (
                q - q.mean(-1, keepdim=True) - xhat * (q * xhat).mean(-1, keepdim=True))
            grad_x[a:b] = g
            if dropout:
                g = g * (_keep(a, b - a, hidden, seed, index * _increment(hidden), p) * scale)
            grad_branch[a:b] = g
            grad_weight += (gy * xhat).sum(0)
            grad_bias += gy.sum(0)
        upstream = grad_x
        gradients.append((grad_x, grad_branch, grad_weight, grad_bias))
    gradients.reverse()
    if case["kind"] == "buffers":
        out = forward[0]
        grad_x, grad_branch, grad_weight, grad_bias = gradients[0]
        return dict(out, mask=None, grad_x=grad_x, grad_branch=grad_branch,
                    grad_weight=grad_weight, grad_bias=grad_bias)
    answer = [current, *(out["normalized"] for out in forward), gradients[0][0]]
    for _, grad_branch, grad_weight, grad_bias in gradients:
        answer.append(grad_branch)
        if not case["frozen"]:
            answer += [grad_weight, grad_bias]
    return answer
