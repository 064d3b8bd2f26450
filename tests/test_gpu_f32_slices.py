"""Single-precision products, whole and with the reduction in slices (nmg_gemm_f32_splitk), against fp64."""
import ctypes

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

import sten_amd as sten
from sten_amd import native

DEV = "cuda:0"
# Sums of a slice are rounded once per 16 positions and once per slice: 2^-24 * sqrt(K / 16 + slices) of the result in 2-norm on N(0, 1)
# data, 9e-7 at K = 4096, if every rounding were of the full sum; the three-part operands leave out 2^-24 at most.
BOUND = 1e-6


def _product(form, A, X, O, K, T, slices, bias=None, pad=0):
    L = native.load()
    Y = torch.full((T, O + pad), 7.0, device=DEV)
    part = torch.full((slices * T * ((O + 3) // 4 * 4),), float("nan"), device=DEV)
    native.check(L.nmg_gemm_f32_splitk(A.data_ptr(), A.stride(0), X.data_ptr(), X.stride(0), Y.data_ptr(), O + pad,
                                       None if bias is None else bias.data_ptr(), O, K, T, form, slices, part.data_ptr(),
                                       part.numel() * 4, native.stream_ptr(A.device)))
    if pad:
        assert torch.all(Y[:, O:] == 7.0)
    return Y[:, :O]


def _operands(form, O, K, T, pad):
    g = torch.Generator(DEV).manual_seed(O + K + T)
    A = torch.randn(*((O, K + pad) if form == 0 else (K, O + pad)), device=DEV, generator=g)
    X = torch.randn(*((T, K + pad) if form < 2 else (K, T + pad)), device=DEV, generator=g)
    a = A[:, :K] if form == 0 else A[:, :O].t()
    x = X[:, :K] if form < 2 else X[:, :T].t()
    return A, X, a, x


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("O,K,T,slices,pad", [
    (128, 256, 128, 2, 0),      # whole tiles and steps
    (96, 96, 96, 3, 0),         # a step a slice
    (4, 65, 5, 3, 3),           # the smallest extents; the last slice is one position
    (129, 1000, 131, 4, 1),     # one past a tile, last slice with an end inside a step, odd pitches
    (250, 2047, 130, 16, 5),
    (1021, 2047, 1999, 2, 0),
    (97, 130, 1024, 5, 2),      # tiles of 96 outputs
])
def test_slices_against_fp64(form, O, K, T, slices, pad):
    print(f"case f32 slices form={form} O={O} K={K} T={T} slices={slices} pad={pad}", flush=True)
    A, X, a, x = _operands(form, O, K, T, pad)
    bias = torch.randn(O, device=DEV) if form == 0 else None
    ref = x.double() @ a.double().t() + (0 if bias is None else bias.double())
    y = _product(form, A, X, O, K, T, slices, bias, pad)
    assert ((y.double() - ref).norm() / ref.norm()).item() <= BOUND


# Whole products with ends inside steps and groups of four: one step fewer than the loop for whole steps takes, as many, and several
# turns of it, on tiles of 32 x 32 (steps of 64; up to one and more than one a CU), 64 x 64 (16) and larger ones, 128 x 96 among them.  On the fp32 instruction sums are rounded once per 2 positions.
@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("O,K,T", [(36, 511, 221), (37, 513, 222), (36, 1618, 221), (1001, 127, 640), (1000, 131, 641), (1000, 383, 639),
                                   (383, 263, 1281), (2664, 279, 263), (1283, 515, 510),
                                   (2085, 515, 209), (1652, 145, 1576)])
def test_whole_products_with_ends_against_fp64(form, O, K, T):
    print(f"case f32 ends form={form} O={O} K={K} T={T}", flush=True)
    A, X, a, x = _operands(form, O, K, T, 0)
    ref = x.double() @ a.double().t()
    y = _product(form, A, X, O, K, T, 1)
    assert ((y.double() - ref).norm() / ref.norm()).item() <= 2.0 ** -24 * (K / 2) ** 0.5


@pytest.mark.gpu
def test_equal_rows_have_equal_sums_and_infinities_stay_in_theirs():
    O, K, T, slices = 200, 700, 300, 3
    A, X, a, x = _operands(0, O, K, T, 0)
    X[137] = X[3]
    X[5, 650] = float("inf")      # (the last slice)
    X[6, 10] = float("nan")
    X[7, 300] = 1e38              # no finite bf16 number after the scaling
    A[11, 20] = 3e38
    y = _product(0, A, X, O, K, T, slices)
    assert torch.equal(y[137], y[3])
    ref = (x.double() @ a.double().t()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
    ok = torch.isfinite(ref)
    rows = (y - ref).double().masked_fill(~ok, 0).norm(dim=1) / ref.double().masked_fill(~ok, 0).norm(dim=1).clamp_min(1e-30)
    assert rows[torch.arange(T, device=DEV) != 6].max().item() <= 4 * BOUND      # (row 6 is NaN throughout; large numbers: fp32 instruction)


def test_the_plan_leaves_no_slice_empty_and_sizes_its_workspace():
    L = native.load()
    seen = set()
    for form in (0, 1, 2):
        for O in (4, 100, 256, 768, 1021, 4096):
            for K in (1, 31, 400, 2047, 4096, 40000):
                for T in (1, 17, 136, 512, 1999, 70000):
                    slices, size = ctypes.c_int(), ctypes.c_int64()
                    native.check(L.nmg_gemm_f32_plan(K if form == 0 else O, T if form == 2 else K, O, K, T, form, ctypes.byref(slices),
                                                     ctypes.byref(size)))
                    s, steps = slices.value, (K + 31) // 32
                    seen.add(s)
                    assert 1 <= s <= 16 and (s - 1) * ((steps + s - 1) // s) < steps
                    assert size.value == (0 if s == 1 else s * T * ((O + 3) // 4 * 4) * 4)
    assert 1 in seen and len(seen) > 3
    # tiles that walk in steps of 16 have no ends with these reductions: as fast whole (23 us, 32 and 29 in slices)
    for form, O, K, T, cut in ((2, 2392, 1168, 264, False), (0, 2016, 1296, 352, False), (2, 2064, 976, 240, False), (0, 768, 3072, 1024, True)):
        native.check(L.nmg_gemm_f32_plan(K if form == 0 else O, T if form == 2 else K, O, K, T, form, ctypes.byref(slices), ctypes.byref(size)))
        assert (slices.value > 1) == cut
    assert L.nmg_gemm_f32_plan(8, 8, -1, 8, 8, 0, ctypes.byref(slices), ctypes.byref(size)) != 0
    assert L.nmg_gemm_f32_plan(8, 8, 8, 8, 8, 3, ctypes.byref(slices), ctypes.byref(size)) != 0


def _sums_of_slices(call):
    """The call's result, and how many of its products came in slices (None where the profiler reports no kernels)."""
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        out = call()
        torch.cuda.synchronize()
    names = [e.name for e in p.events() if "nmg::" in e.name]
    return out, sum("splitk_sum_kernel<float" in n for n in names) if names else None


def _close(got, ref, name):
    assert got.shape == ref.shape
    assert ((got.double() - ref).norm() / ref.norm()).item() <= BOUND, name
    # every element: BOUND of the root mean square is a standard deviation of those roundings, eight of them
    assert (got.double() - ref).abs().max().item() <= 8 * BOUND * ref.pow(2).mean().sqrt().item(), name


# The public calls whose products are in slices, one of the three in each case: forward with a bias, gradient of the input, of the weight, and the
# same of torch.mm; operands with a pitch and an offset of their own, whole extents and odd ones.
@pytest.mark.gpu
@pytest.mark.parametrize("O,K,T", [(768, 3072, 1024), (3072, 768, 1024), (768, 1024, 3072), (767, 3071, 1021), (3071, 767, 1021), (767, 1021, 3071)])
def test_public_calls_in_slices(O, K, T):
    print(f"case f32 slices, public calls O={O} K={K} T={T}", flush=True)
    g = torch.Generator(DEV).manual_seed(O)
    lin = torch.nn.Linear(K, O, device=DEV)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(O, K, device=DEV, generator=g))
        lin.bias.copy_(torch.randn(O, device=DEV, generator=g))
    sb = sten.SparsityBuilder()
    sb.set_weight("weight", initial_sparsifier=sten.GroupedNMSparsifier(2, 4, 16, sparse_dim=1, group_dim=0), out_format=sten.GroupedNMTensor)
    lin = sb.sparsify_model_inplace(lin)
    W = lin.weight.wrapped_tensor.to_dense().double()

    def strided(rows, cols):
        wide = torch.randn(rows, cols + 6, device=DEV, generator=g)
        return wide[:, 3:3 + cols]

    x, gy = strided(T, K), strided(T, O)

    def train():
        lin.zero_grad(set_to_none=True)
        leaf = x.detach().requires_grad_(True)
        y = lin(leaf)
        y.backward(gy)
        return y.detach(), leaf.grad, lin.weight.grad.wrapped_tensor.to_dense()

    (y, gx, gw), sums = _sums_of_slices(train)
    assert sums in (None, 1), "the plan gives no slices: other extents"
    _close(y, x.double() @ W.t() + lin.bias.detach().double(), "linear")
    _close(gx, gy.double() @ W, "gradient of the input")
    _close(gw, gy.double().t() @ x.double(), "gradient of the weight")

    b, gc = strided(K, T), strided(O, T)

    def mm():
        lin.zero_grad(set_to_none=True)
        leaf = b.detach().requires_grad_(True)
        c = torch.mm(lin.weight, leaf)
        c.backward(gc)
        return c.detach(), leaf.grad, lin.weight.grad.wrapped_tensor.to_dense()

    (c, gb, gw), sums = _sums_of_slices(mm)
    assert sums in (None, 1), "the plan gives no slices: other extents"
    _close(c, W @ b.double(), "mm")
    _close(gb, W.t() @ gc.double(), "gradient of B")
    _close(gw, gc.double() @ b.double().t(), "gradient of the weight of mm")
