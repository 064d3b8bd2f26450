"""16-bit products at extents that are no whole K steps, pieces of 8 elements or 16-byte rows: forward, both gradients
and torch.mm against float64, and the copy that brings operands into shape."""
import numpy as np
import pytest
import torch

import sten_amd as sten
from sten_amd import native
from helpers import rel_l2, seeded, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float16: 1e-3, torch.bfloat16: 8e-3}


@pytest.mark.parametrize("rows,cols,pitch,drows,dcols,dpitch", [
    (1, 1, 1, 1, 8, 8), (3, 7, 7, 3, 64, 64), (5, 1001, 1003, 8, 1024, 1024), (17, 64, 65, 64, 64, 64), (4, 72, 72, 3, 69, 71), (0, 8, 8, 2, 8, 8)])
def test_copy_rows(rows, cols, pitch, drows, dcols, dpitch):
    src = torch.zeros(max(rows, 1), pitch, dtype=torch.float16, device=DEV)
    src[:rows, :cols] = seeded((rows, cols), torch.float16, seed=3).to(DEV)
    dst = torch.full((drows, dpitch), 7.0, dtype=torch.float16, device=DEV)
    native.check(native.load().nmg_copy_rows16(native.ptr(src), rows, cols, pitch, native.ptr(dst), drows, dcols, dpitch, None))
    want = torch.full((drows, dpitch), 7.0, dtype=torch.float16)
    want[:, :dcols] = 0
    r, c = min(rows, drows), min(cols, dcols)
    want[:r, :c] = src[:r, :c].cpu()
    assert torch.equal(dst.cpu(), want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C,T", [(67, 65, 5), (65, 130, 17), (129, 1001, 33), (300, 520, 70), (257, 191, 129), (1030, 515, 1)])
@pytest.mark.parametrize("n,m,g", [(2, 4, 4), (2, 8, 2), (4, 8, 1), (3, 6, 2)])
@pytest.mark.parametrize("along", [0, 1])
def test_odd_extents(R, C, T, n, m, g, along, dtype):
    print(f"case {R}x{C} T={T} {n}:{m}:{g} along={along} {dtype}", flush=True)
    w = sten.GroupedNMTensor.from_dense(seeded((R, C), dtype, seed=1, std=0.5).to(DEV), n, m, sparse_dim=along, group_size=g,
                                        group_dim=1 - along)
    Wd = to_np(w.to_dense()).astype(np.float64)
    x, gy = seeded((T, C), dtype, seed=2), seeded((T, R), dtype, seed=3)
    X, G = to_np(x).astype(np.float64), to_np(gy).astype(np.float64)
    y = sten.spmm(w, x.to(DEV), reduce_dim=1)
    assert rel_l2(to_np(y), X @ Wd.T) <= TOL[dtype]
    gx = sten.spmm(w, gy.to(DEV), reduce_dim=0)
    assert rel_l2(to_np(gx), G @ Wd) <= TOL[dtype]
    mask = (to_np(w.clone_layout(torch.ones(R, C, dtype=dtype, device=DEV)).to_dense()) != 0)
    for kw in ({}, {"reduction_last": True}) if T % 8 == 0 else ({},):
        a, b = (gy.to(DEV), x.to(DEV)) if not kw else (gy.t().contiguous().to(DEV), x.t().contiguous().to(DEV))
        gw = w.masked_product(a, b, **kw)
        assert rel_l2(to_np(gw.to_dense()), (G.T @ X) * mask) <= TOL[dtype]
    sp = sten.SparseTensorWrapper.wrapped_from_dense(w, w.to_dense(), None)
    sp.grad_fmt = (sten.KeepAll(), sten.GroupedNMTensor, sten.KeepAll(), sten.GroupedNMTensor)
    leaf = torch.nn.Parameter(sp) if isinstance(sp, torch.nn.Parameter) else sp.requires_grad_(True)
    b = x.t().contiguous().to(DEV).requires_grad_(True)
    c = torch.mm(leaf, b)
    assert c.shape == (R, T) and rel_l2(to_np(c), Wd @ X.T) <= TOL[dtype]
    c.backward(gy.t().contiguous().to(DEV))
    assert rel_l2(to_np(b.grad), (G @ Wd).T) <= TOL[dtype]
    assert rel_l2(to_np(leaf.grad.wrapped_tensor.to_dense()), (G.T @ X) * mask) <= TOL[dtype]
    from sten_amd.impls import _dense_product
    gd = _dense_product("tn", gy.to(DEV), x.to(DEV))
    assert gd.shape == (R, C) and rel_l2(to_np(gd), G.T @ X) <= TOL[dtype]
    gn = _dense_product("nt", gy.t().contiguous().to(DEV), x.t().contiguous().to(DEV))
    assert gn.shape == (R, C) and rel_l2(to_np(gn), G.T @ X) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,T", [(3, 17), (1021, 20), (1028, 33), (2050, 130)])
@pytest.mark.parametrize("slices", [2, 3, 8, 16])      # 16 steps: none leaves a slice empty
def test_sum_of_slices(R, T, slices, dtype):
    w = sten.GroupedNMTensor.from_dense(seeded((R, 1024), dtype, seed=1, std=0.5).to(DEV), 2, 4, sparse_dim=0, group_size=4, group_dim=1)
    x, bias = seeded((T, 1024), dtype, seed=2), seeded((R,), dtype, seed=3)
    w.spmm_opt["slices"] = slices
    y = sten.spmm(w, x.to(DEV), bias.to(DEV), reduce_dim=1)
    want = to_np(x).astype(np.float64) @ to_np(w.to_dense()).astype(np.float64).T + to_np(bias).astype(np.float64)
    assert rel_l2(to_np(y), want) <= TOL[dtype]
