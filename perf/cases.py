"""What the framework is measured on: the work that its users give it, through its public entry points.

A case is one layer or one weight with everything that a program holds around it:
  linear    forward of a sparse ``torch.nn.Linear`` without gradients -- serving: a few tokens while
            text is generated, hundreds to thousands while a prompt is read
  int4      the same on the 2:4 + int4 weight, which exists for generation with a few tokens
  train     forward, backward and SGD step of a sparse ``torch.nn.Linear``
  mm        ``torch.mm(W, B)`` with a sparse W, forward and backward
  sparsify  a dense weight into the grouped n:m format -- on loading a model, and whenever a
            training schedule chooses the pattern anew

``along`` says where the n:m blocks lie: "outputs" is what ``GroupedNMSparsifier(n, m, g)`` gives (the
default), "inputs" is the orientation that the sparse matrix cores can use in forward.
``rows`` x ``cols`` is the weight ([out_features, in_features]); ``tokens`` the rows of the
activations (the columns of B for ``mm``).
"""
import math

import torch

import sten_amd as sten

DEVICE = "cuda:0"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ITEM = {"f16": 2, "bf16": 2, "f32": 4}
PATTERNS = ((2, 4, 16), (1, 8, 32), (2, 8, 32), (4, 8, 32), (3, 6, 12))
LEARNING_RATE = 1e-3


def _case(name, kind, rows, cols, tokens, dtype, pattern, along, bias=False, grad="dense"):
    n, m, g = pattern
    c = {"kind": kind, "rows": rows, "cols": cols, "tokens": tokens, "dtype": dtype, "n": n, "m": m, "g": g,
         "along": along, "bias": bias, "grad": grad}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one generated token through a down-projection: the latency of a serving loop
        _case("decode_1", "linear", 4096, 11008, 1, "f16", (2, 4, 16), "inputs"),
        # sixteen sequences generated together through an up-projection, default orientation
        _case("decode_16_default", "linear", 11008, 4096, 16, "bf16", (2, 4, 16), "outputs"),
        # four sequences on the int4 format
        _case("decode_4_int4", "int4", 11008, 4096, 4, "f16", (2, 4, 1), "inputs"),
        # a prompt of 2048 tokens: the headline product
        _case("prefill_2048", "linear", 4096, 11008, 2048, "f16", (2, 4, 16), "inputs"),
        # a prompt of no particular length, a dense pattern, default orientation, with a bias
        _case("prefill_ragged_default", "linear", 4096, 4096, 777, "bf16", (4, 8, 32), "outputs", bias=True),
        # a small single-precision projection: launches and the host path
        _case("small_f32", "linear", 768, 768, 256, "f32", (2, 4, 16), "inputs", bias=True),
        # a feed-forward layer in single precision over a batch of sequences
        _case("batch_f32", "linear", 768, 3072, 4096, "f32", (3, 6, 12), "outputs"),
        # fine-tuning a small layer with every default: orientation, dense gradient, bias
        _case("train_small_f32", "train", 768, 3072, 512, "f32", (2, 4, 16), "outputs", bias=True),
        # training a large layer with the gradient in the weight's own pattern
        _case("train_large", "train", 16384, 4096, 4096, "f16", (2, 4, 16), "inputs", grad="pattern"),
        # the matrix product as an operator of its own, both gradients
        _case("mm_2048", "mm", 4096, 4096, 2048, "f16", (2, 4, 16), "inputs"),
        # sparsifying one layer of a model ...
        _case("sparsify_2_4", "sparsify", 4096, 4096, 0, "f16", (2, 4, 16), "inputs"),
        # ... and a large one with a pattern of many columns per tile, default orientation
        _case("sparsify_2_8_default", "sparsify", 8192, 8192, 0, "f16", (2, 8, 32), "outputs"),
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _extent(rng, low, high, step):
    return max(step, _log_uniform(rng, low, high) // step * step)


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "int4", "train", "train", "mm", "sparsify", "sparsify"))
    # most layers have extents that are multiples of 128; vocabularies and pruned layers do not
    step = rng.choice((128, 128, 128, 8, 8, 1))
    along = rng.choice(("inputs", "outputs"))
    if kind == "int4":      # the format takes in_features in multiples of 128
        return _case(None, kind, _extent(rng, 1024, 16384, step), _extent(rng, 1024, 8192, 128),
                     _log_uniform(rng, 1, 16), "f16", (2, 4, 1), "inputs", bias=rng.random() < 0.5)
    dtype = rng.choice(("f16", "bf16", "f32"))
    pattern = rng.choice(PATTERNS)
    if kind == "sparsify":
        rows = _extent(rng, 512, 8192, step)
        most = (2 ** 24 if pattern[:2] == (4, 8) else 2 ** 26) // (2 if dtype == "f32" else 1)
        return _case(None, kind, rows, _extent(rng, 512, max(512, min(8192, most // rows)), step), 0, dtype, pattern, along)
    low, high = (256, 4096) if dtype == "f32" else (512, 16384)
    rows = _extent(rng, low, high, step)
    cols = _extent(rng, low, max(low, min(high, 2 ** 26 // rows)), step)
    # single precision runs at a sixteenth of the 16-bit rate, odd extents and three products cost more than one
    most = 2 ** 33 if dtype == "f32" or step == 1 else 2 ** 36
    most //= 1 if kind == "linear" else 4
    tokens = _log_uniform(rng, 1, 16) if kind == "linear" and rng.random() < 0.5 else _log_uniform(rng, 17, 4096)
    return _case(None, kind, rows, cols, max(1, min(tokens, most // (rows * cols))), dtype, pattern, along,
                 bias=kind != "mm" and rng.random() < 0.5,
                 grad=rng.choice(("dense", "pattern")) if kind in ("train", "mm") else "dense")


def _randn(gen, *shape, dtype, scale=1.0):
    return (torch.randn(*shape, generator=gen, device=DEVICE) * scale).to(dtype)


def _sparsifier(case):
    if case["along"] == "outputs":
        return sten.GroupedNMSparsifier(case["n"], case["m"], case["g"])
    return sten.GroupedNMSparsifier(case["n"], case["m"], case["g"], sparse_dim=-1, group_dim=-2)


def _builder(case, initial_sparsifier, out_format):
    builder = sten.SparsityBuilder()
    builder.set_weight("weight", initial_sparsifier=initial_sparsifier, out_format=out_format)
    if case["grad"] == "pattern":
        builder.set_weight_grad("weight", tmp_format=sten.GroupedNMTensor, out_format=sten.GroupedNMTensor)
    return builder


def prepare(case, seed):
    gen = torch.Generator(DEVICE).manual_seed(seed)
    dtype, rows, cols, tokens = DTYPES[case["dtype"]], case["rows"], case["cols"], case["tokens"]
    weight = _randn(gen, rows, cols, dtype=dtype, scale=0.02)
    state = {"case": dict(case)}
    if case["kind"] == "sparsify":
        state["weight"] = weight
        return state
    layer = torch.nn.Linear(cols, rows, bias=case["bias"], device=DEVICE, dtype=dtype)
    with torch.no_grad():
        layer.weight.copy_(weight)
        if case["bias"]:
            layer.bias.copy_(_randn(gen, rows, dtype=dtype, scale=0.02))
    del weight
    if case["kind"] == "int4":
        builder = _builder(case, sten.SparseMarlinSparsifier(), sten.SparseMarlinTensor)
    else:
        builder = _builder(case, _sparsifier(case), sten.GroupedNMTensor)
    layer = builder.sparsify_model_inplace(layer)
    state["layer"] = layer
    if case["kind"] == "mm":
        state["input"] = _randn(gen, cols, tokens, dtype=dtype).requires_grad_(True)
        state["grad"] = _randn(gen, rows, tokens, dtype=dtype, scale=0.01)
        return state
    state["input"] = _randn(gen, tokens, cols, dtype=dtype)
    if case["kind"] == "train":
        state["input"].requires_grad_(True)      # a layer inside a network: the gradient goes on to the one before
        state["grad"] = _randn(gen, tokens, rows, dtype=dtype, scale=0.01)
        state["optimizer"] = torch.optim.SGD(layer.parameters(), lr=LEARNING_RATE)
    return state


def _weight_grad(weight):
    grad = weight.grad.wrapped_tensor
    return grad.val if isinstance(grad, sten.GroupedNMTensor) else grad.to_dense()


def run(state):
    case = state["case"]
    if case["kind"] == "sparsify":
        dims = (0, 1) if case["along"] == "outputs" else (1, 0)
        sparse = sten.GroupedNMTensor.from_dense(state["weight"], case["n"], case["m"], sparse_dim=dims[0],
                                                 group_size=case["g"], group_dim=dims[1])
        return {"val": sparse.val, "idx": sparse.idx}
    layer, x = state["layer"], state["input"]
    if case["kind"] in ("linear", "int4"):
        with torch.no_grad():
            return layer(x)
    x.grad = None
    if case["kind"] == "mm":
        layer.weight.grad = None
        y = torch.mm(layer.weight, x)
        y.backward(state["grad"])
        return {"y": y.detach(), "grad_input": x.grad, "grad_weight": _weight_grad(layer.weight)}
    state["optimizer"].zero_grad(set_to_none=True)
    y = layer(x)
    y.backward(state["grad"])
    state["optimizer"].step()
    out = {"y": y.detach(), "grad_input": x.grad, "grad_weight": _weight_grad(layer.weight),
           "weight": layer.weight.wrapped_tensor.val}
    if case["bias"]:
        out.update(grad_bias=layer.bias.grad, bias=layer.bias.detach())
    return out


def work(case):
    item, rows, cols, tokens = ITEM[case["dtype"]], case["rows"], case["cols"], case["tokens"]
    n, m = case["n"], case["m"]
    dense, product = rows * cols, 2.0 * rows * cols * tokens
    kept, blocks = dense * n / m, dense / m
    acts, outs, bias = tokens * cols * item, tokens * rows * item, rows * item if case["bias"] else 0
    if case["kind"] == "int4":      # half a byte a kept value, 2 bits of position, a scale for 128 positions
        return {"bytes": kept / 2 + kept / 4 + dense / 128 * 2 + acts + outs + bias, "flops": product * n / m}
    compressed = kept * item + blocks * 2
    if case["kind"] == "sparsify":
        return {"bytes": dense * item + compressed, "flops": 0}
    if case["kind"] == "linear":
        return {"bytes": compressed + acts + outs + bias, "flops": product * n / m}
    # forward and the input's gradient on the kept values; the weight's gradient on what it stores
    grad = dense if case["grad"] == "dense" else kept
    total = compressed + 2 * acts + 2 * outs + grad * item
    if case["kind"] == "train":
        total += kept * item + 3 * bias      # the updated weight; the bias, its gradient and its update
    return {"bytes": total, "flops": product * (2 * n / m + grad / dense)}


def tolerance(case):
    if case["kind"] == "sparsify":
        return "exact"
    return {"rel": {"f32": 1e-5, "f16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
