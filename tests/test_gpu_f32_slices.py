"""Single-precision products, whole and with the reduction in slices (nmg_gemm_f32_splitk), against fp64."""
import ctypes

import pytest
import torch

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
# turns of it, on tiles of 32 x 32 (steps of 64), 64 x 64 (16) and larger ones.  On the fp32 instruction sums are rounded once per 2 positions.
@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1, 2])
@pytest.mark.parametrize("O,K,T", [(36, 511, 221), (37, 513, 222), (36, 1618, 221), (1001, 127, 640), (1000, 131, 641), (1000, 383, 639),
                                   (383, 263, 1281), (2664, 279, 263), (1283, 515, 510)])
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
    assert L.nmg_gemm_f32_plan(8, 8, -1, 8, 8, 0, ctypes.byref(slices), ctypes.byref(size)) != 0
    assert L.nmg_gemm_f32_plan(8, 8, 8, 8, 8, 3, ctypes.byref(slices), ctypes.byref(size)) != 0
