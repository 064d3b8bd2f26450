"""A product with a bias is rounded once, whichever kernel computes it."""
import numpy as np
import pytest
import torch

import sten_amd as sten
from helpers import to_np
from sten_amd import native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def whole(shape, dtype, seed):
    return torch.randint(-30, 31, shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def rounded_once(y, exact, dtype):
    # whole numbers up to 30: partial sums of up to 4224 products and the bias are below 2^24 and exact in single
    # precision in any order; the one rounding is off by u = 2^-11 of a value in fp16, 2^-8 in bf16.  Most sums are
    # beyond 2048 and 256, so that one more rounding before the bias is added shows
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    return (np.abs(to_np(y).astype(np.float64) - exact) <= u * np.abs(exact)).all()


def f64(t):
    return to_np(t).astype(np.float64)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C,T,n,m,g,rd,kernel,opt", [
    (300, 512, 130, 2, 4, 16, 1, "smfmac", {"slices": 1}),       # the tile by itself: 128 x 128
    (300, 512, 130, 2, 4, 16, 1, "smfmac", {"variant": 0}),
    (300, 512, 130, 2, 4, 16, 1, "smfmac", {"variant": 6}),      # 256 x 128, 256 x 256
    (300, 512, 260, 2, 4, 16, 1, "smfmac", {"variant": 8}),
    (300, 512, 130, 2, 4, 16, 1, "smfmac", {"slices": 3}),
    (300, 512, 16, 2, 4, 16, 1, "smfmac", {"variant": 5}),
    (300, 512, 130, 4, 8, 4, 1, "densefrag", {"slices": 1}),
    (300, 512, 130, 4, 8, 4, 1, "densefrag", {"dense_variant": 0}),
    (300, 512, 260, 4, 8, 4, 1, "densefrag", {"dense_variant": 1}),
    (300, 512, 130, 4, 8, 4, 1, "densefrag", {"slices": 3}),
    (512, 301, 130, 2, 4, 16, 0, "densefrag", {"slices": 1}),    # outputs along the sparse dim
    (300, 512, 130, 4, 8, 4, 1, "mfma", {"expand": False}),      # weights expanded inside the kernel
    (512, 304, 130, 2, 4, 16, 0, "mfma", {"expand": False}),
    (300, 512, 130, 4, 8, 4, 1, "expand", {}),                   # a dense copy, then the product of rows
    (300, 512, 1, 2, 4, 16, 1, None, {}),                        # few tokens
    (301, 512, 9, 2, 4, 16, 0, None, {}),
    (512, 300, 3, 2, 4, 16, 0, None, {}),
])
def test_products(dtype, R, C, T, n, m, g, rd, kernel, opt):
    print(f"case {dtype} {R}x{C} T={T} {n}:{m}:{g} reduce_dim={rd} {kernel} {opt}", flush=True)
    w = sten.GroupedNMTensor.from_dense(whole((R, C), dtype, 1).to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
    w.spmm_opt.update(opt)
    D = f64(w.to_dense())
    x = whole((T, C if rd == 1 else R), dtype, 2)
    bias = whole((R if rd == 1 else C,), dtype, 3)
    y = sten.spmm(w, x.to(DEV), bias.to(DEV), reduce_dim=rd, kernel=kernel)
    assert rounded_once(y, f64(x) @ (D.T if rd == 1 else D) + f64(bias), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form,N", [("ct", 100), ("ct", 200), ("ct", 4000), ("tt", 200)])
@pytest.mark.parametrize("n,m", [(2, 4), (4, 8)])
def test_transposed_results(dtype, form, N, n, m):
    """C [R, N] = W B + bias per row, on the sparse and the dense cores."""
    R, C = 4100 if N == 4000 else 300, 512
    print(f"case {dtype} {form} N={N} {n}:{m}", flush=True)
    w = sten.GroupedNMTensor.from_dense(whole((R, C), dtype, 1).to(DEV), n, m, sparse_dim=1, group_size=4, group_dim=0)
    B, bias = whole((C, N), dtype, 2).to(DEV), whole((R,), dtype, 3).to(DEV)
    operand = w.fragpack() if m == 4 else (w.densefrag(1),)
    x, ldx = (B, N) if form == "tt" else (B.t().contiguous(), C)
    out = torch.empty(R, N, dtype=dtype, device=DEV)
    entry = getattr(native.load(), ("nmg_spmm_smfmac_" if m == 4 else "nmg_spmm_densefrag_") + form)
    native.check(entry(*[native.ptr(t) for t in operand], R, C, native.ptr(x), ldx, native.ptr(out), N, native.ptr(bias), N,
                       native.dtype_code(dtype), None))
    assert rounded_once(out, f64(w.to_dense()) @ f64(B) + f64(bias)[:, None], dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form,O,K,T", [
    ("nt", 300, 512, 130),       # 256 x 128
    ("nt", 4000, 512, 4090),     # 256 x 256
    ("tn", 296, 500, 136),
    ("tn", 8, 500, 264),
])
def test_dense_products(dtype, form, O, K, T):
    print(f"case {dtype} {form} {O} {K} {T}", flush=True)
    a, x = (whole((O, K), dtype, 1), whole((T, K), dtype, 2)) if form == "nt" else (whole((K, O), dtype, 1), whole((K, T), dtype, 2))
    bias = whole((O,), dtype, 3)
    A, X, b, y = a.to(DEV), x.to(DEV), bias.to(DEV), torch.empty(T, O, dtype=dtype, device=DEV)
    native.check(getattr(native.load(), "nmg_gemm_" + form)(native.ptr(A), a.shape[1], native.ptr(X), x.shape[1], native.ptr(y), O, native.ptr(b),
                                                            O, K, T, native.dtype_code(dtype), None))
    exact = f64(x) @ f64(a).T if form == "nt" else f64(x).T @ f64(a)
    assert rounded_once(y, exact + f64(bias), dtype)
