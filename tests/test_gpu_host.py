"""The native dispatch of wrapped weights (csrc/nmg_host.cpp) against the Python dispatcher, which stays the
route of every other call: same kernels, so the same bits."""
import pytest
import torch
import torch.nn.functional as F

import sten_amd as sten
from sten_amd import dispatch, native
from helpers import rel_l2, seeded, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def weight(dtype, grad):
    layer = torch.nn.Linear(128, 96, bias=True, device=DEV, dtype=dtype)
    with torch.no_grad():
        layer.weight.copy_(seeded((96, 128), dtype, seed=1, std=0.1).to(DEV))
    builder = sten.SparsityBuilder()
    builder.set_weight("weight", initial_sparsifier=sten.GroupedNMSparsifier(2, 4, 4), out_format=sten.GroupedNMTensor)
    if grad == "pattern":
        builder.set_weight_grad("weight", tmp_format=sten.GroupedNMTensor, out_format=sten.GroupedNMTensor)
    return builder.sparsify_model_inplace(layer)


def results(call, layer, x, shape):
    x.grad = layer.weight.grad = layer.bias.grad = None
    y = call()
    y.backward(seeded(shape, x.dtype, seed=3).to(DEV))
    g = layer.weight.grad.wrapped_tensor
    out = [y.detach(), x.grad, g.val if isinstance(g, sten.GroupedNMTensor) else g.to_dense()]
    return out + ([] if layer.bias.grad is None else [layer.bias.grad])


@pytest.mark.parametrize("grad", ["dense", "pattern"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("op,lead", [("linear", (1,)), ("linear", (33,)), ("linear", (3, 5)), ("nobias", (17,)), ("mm", (40,))])
def test_native_dispatch_gives_what_the_python_dispatcher_gives(op, lead, dtype, grad):
    print(f"case {op} {lead} {dtype} {grad}", flush=True)
    layer = weight(dtype, grad)
    if op == "mm":
        x = seeded((128, 40), dtype, seed=2).to(DEV).requires_grad_(True)
        func, args, shape = torch.mm, (layer.weight, x), (96, 40)
    else:
        x = seeded(lead + (128,), dtype, seed=2).to(DEV).requires_grad_(True)
        func, args, shape = F.linear, (x, layer.weight) + ((layer.bias,) if op == "linear" else ()), lead + (96,)
    native = results(lambda: func(*args), layer, x, shape)
    python = results(lambda: dispatch._torch_function(func, (), args, None), layer, x, shape)
    assert len(native) == len(python)
    for a, b in zip(native, python):
        assert a.shape == b.shape and torch.equal(a, b)


def test_a_graph_is_walked_once():
    layer = weight(torch.float32, "dense")
    y = layer(seeded((4, 128), torch.float32, seed=2).to(DEV))
    y.sum().backward()
    with pytest.raises(RuntimeError):
        y.sum().backward()


def test_transforms_reach_the_python_dispatcher():
    """Forward-mode tangents and function transforms: refused there, never dropped."""
    import torch.autograd.forward_ad as forward_ad
    layer = weight(torch.float32, "dense")
    x = seeded((4, 128), torch.float32, seed=2).to(DEV)
    with forward_ad.dual_level():
        with pytest.raises(NotImplementedError):
            layer(forward_ad.make_dual(x, torch.ones_like(x)))
        bias = forward_ad.make_dual(layer.bias.detach(), torch.ones_like(layer.bias))
        with pytest.raises(NotImplementedError):
            F.linear(x, layer.weight, bias)
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.vmap(layer)(x.reshape(2, 2, 128))
    with pytest.raises(RuntimeError, match="functorch"):
        torch.func.grad(lambda v: layer(v).sum())(x)
    assert layer(x).shape == (4, 96)


class Product(torch.nn.Module):
    """One operator on a sparse weight, with the weight (and bias) of ``layer``."""

    def __init__(self, layer, op):
        super().__init__()
        self.weight, self.bias, self.op = layer.weight, layer.bias, op

    def forward(self, x):
        if self.op == "mm":
            return torch.mm(self.weight, x)
        return F.linear(x, self.weight, self.bias if self.op == "linear" else None)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("op", ["linear", "nobias", "mm", "int4"])
def test_a_traced_module_computes(op, grad):
    """torch.jit.trace of a module: the graph holds the product, not the bare allocation of its result."""
    print(f"case {op} grad={grad}", flush=True)
    if op == "int4":
        layer = torch.nn.Linear(128, 96, device=DEV, dtype=torch.float16)
        builder = sten.SparsityBuilder()
        builder.set_weight("weight", initial_sparsifier=sten.SparseMarlinSparsifier(), out_format=sten.SparseMarlinTensor)
        module = Product(builder.sparsify_model_inplace(layer).requires_grad_(False), "linear")
    else:
        module = Product(weight(torch.float16, "dense").requires_grad_(grad), op)
    shape = (128, 40) if op == "mm" else (8, 128)
    first, second = (seeded(shape, torch.float16, seed=s).to(DEV) for s in (4, 5))
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(module, (first,), check_trace=False)
        for x in (second, first):
            assert torch.equal(traced(x), module(x))


def test_kernel_names():
    """A name that there is no kernel of is refused on every route; "" leaves the choice to the weight's options."""
    layer = weight(torch.float16, "dense")
    w = layer.weight.wrapped_tensor
    x = seeded((4, 128), torch.float16, seed=6).to(DEV)
    want = sten.spmm(w, x, reduce_dim=1)
    for name in ("x", "MFMA", "auto "):
        for reduce_dim in (0, 1):
            with pytest.raises(KeyError, match=name):
                sten.spmm(w, x[:, :w.shape[reduce_dim]].contiguous(), reduce_dim=reduce_dim, kernel=name)
        w.spmm_opt["kernel"] = name
        for call in (lambda: layer(x), lambda: torch.mm(layer.weight, x.t().contiguous())):
            with pytest.raises(KeyError, match=name), pytest.warns(UserWarning, match="Exception raised during handling"):
                call()
        w.spmm_opt["kernel"] = "auto"
    assert torch.equal(sten.spmm(w, x, reduce_dim=1, kernel=""), want)
    for name in native.KERNELS:
        try:
            sten.spmm(w, x, reduce_dim=1, kernel=name)
        except native.NmgError:      # the kernel does not take the shape
            pass


def test_options_are_converted_like_int_does():
    w = weight(torch.float16, "dense").weight.wrapped_tensor
    x = seeded((40, 96), torch.float16, seed=7).to(DEV)
    want = to_np(sten.spmm(w, x, reduce_dim=0))
    for name, value in (("variant", "-1"), ("dense_variant", -1.0), ("slices", "1"), ("slices", -1)):
        w.spmm_opt[name] = value
        assert rel_l2(to_np(sten.spmm(w, x, reduce_dim=0)), want) < 2e-3      # two roundings of the result to 11 bits
        del w.spmm_opt[name]
