"""The direct kernels on the tiles that they take by themselves: 256 x 128, 128 x 128, slices of either, 256 x 256."""
import ctypes

import numpy as np
import pytest
import torch

import sten_amd as sten
from helpers import to_np
from sten_amd import native

DEV = "cuda:0"


def plan(O, K, T, entry="nmg_densefrag_plan"):
    slices, ws = ctypes.c_int(0), ctypes.c_int64(0)
    assert getattr(native.load(), entry)(O, K, T, ctypes.byref(slices), ctypes.byref(ws)) == 0
    return slices.value, ws.value


@pytest.mark.parametrize("entry", ["nmg_densefrag_plan", "nmg_smfmac_plan"])
def test_plan_leaves_no_slice_empty(entry):
    for O in (1, 100, 128, 129, 256, 1000, 4096, 16384, 50000):
        for K in (0, 64, 192, 256, 512, 576, 4096, 11008):
            for T in (0, 1, 17, 128, 129, 777, 4096):
                s, ws = plan(O, K, T, entry)
                steps = K // 64
                assert s == 1 or (2 <= s <= 16 and (s - 1) * -(-steps // s) < steps and steps // s >= 4)
                assert ws == (0 if s == 1 else s * T * -(-O // 256) * 256 * 4)
                if entry == "nmg_smfmac_plan" and T <= 16:
                    assert s == 1
    assert plan(16384, 4096, 4096, entry)[0] == 1 and plan(1024, 16384, 128, entry)[0] > 1 and plan(1024, 1000, 128, entry)[0] == 1
    lib = native.load()
    s, ws = ctypes.c_int(0), ctypes.c_int64(0)
    assert getattr(lib, entry)(-1, 64, 64, ctypes.byref(s), ctypes.byref(ws)) == 1
    assert getattr(lib, entry)(64, 64, 64, None, ctypes.byref(ws)) == 1


def whole(shape, dtype, seed):
    return torch.randint(-3, 4, shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def within(y, prod, bias, dtype):
    # whole numbers up to 3: partial sums of up to 8384 products and the bias are below 2^24 and exact in single precision in any
    # order, so only the one rounding of the result is left: u = 2^-11 of a value in fp16, 2^-8 in bf16
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    return (np.abs(to_np(y).astype(np.float64) - (prod + bias)) <= u * np.abs(prod + bias)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("pattern", [(4, 8, 4), (2, 4, 16)])
@pytest.mark.parametrize("R,C,T,slices", [
    (128, 64, 17, -1),        # one step, fewer than are in flight
    (127, 128, 128, -1),
    (129, 192, 129, -1),      # a last tile of one output and one token
    (255, 256, 300, -1),      # four steps, as many as are in flight
    (33, 320, 130, -1),
    (256, 384, 100, -1),      # six and seven: as in flight on the sparse cores, and one more
    (256, 448, 100, -1),
    (384, 512, 31, -1),       # as many steps as stages
    (1000, 576, 777, -1),     # one more; outputs that are no multiple of 16
    (1640, 1920, 386, -1),
    (4096, 2048, 777, -1),    # 224 of the narrow tiles
    (16384, 256, 200, -1),    # 256 of them
    (2200, 320, 3881, -1),    # several rounds of either tile
    (256, 4224, 40, 2),       # slices of 33 steps
    (300, 4160, 200, 3),      # of 22, 22 and 21
    (129, 8384, 17, 15),      # of 9 and 5 at the end
    (640, 1088, 300, 4),      # of 5, 5, 5 and 2: the last shorter than the steps in flight
    (1100, 4096, 129, -1),    # what the plan takes
])
def test_products_of_every_tile(dtype, pattern, R, C, T, slices):
    n, m, g = pattern
    print(f"case {dtype} {n}:{m} {R}x{C} T={T} slices={slices} plans={plan(R, C, T)} {plan(R, C, T, 'nmg_smfmac_plan')}", flush=True)
    W, x = whole((R, C), dtype, R + C + T), whole((T, C), dtype, 1)
    w = sten.GroupedNMTensor.from_dense(W.to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
    if slices >= 0:
        w.spmm_opt["slices"] = slices
    D = to_np(w.to_dense()).astype(np.float64)
    bias = whole((R,), dtype, 2)
    y = sten.spmm(w, x.to(DEV), bias.to(DEV), reduce_dim=1, kernel="densefrag" if m == 8 else "smfmac")
    prod = to_np(x).astype(np.float64) @ D.T
    assert within(y, prod, to_np(bias).astype(np.float64), dtype)
    if slices < 0:
        # its transposed result
        c = sten.spmm_tt(w, x.to(DEV).t().contiguous())
        assert within(c, prod.T, 0.0, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [(1, 1), (1, 7), (3, 3), (1, 9), (5, 3), (1, 23), (3, 11)])
def test_every_tile_once(tiles):
    # counts of tiles of 256 x 128 with every remainder by the 8 runs that the workgroups are dealt to
    R, C, T = tiles[0] * 256 - 8, 128, tiles[1] * 128 - 4
    for n, m, g, opt in ((2, 4, 16, {"variant": 6}), (2, 4, 16, {"variant": 0}), (4, 8, 4, {"dense_variant": 0})):
        print(f"case {tiles} {n}:{m} {opt}", flush=True)
        W, x = whole((R, C), torch.float16, R), whole((T, C), torch.float16, T)
        w = sten.GroupedNMTensor.from_dense(W.to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
        w.spmm_opt.update(opt)
        prod = to_np(x).astype(np.float64) @ to_np(w.to_dense()).astype(np.float64).T
        y = sten.spmm(w, x.to(DEV), reduce_dim=1, kernel="smfmac" if m == 4 else "densefrag")
        assert within(y, prod, 0.0, torch.float16)
    # the gradient in the weight's own pattern
    w = sten.get_sparsifier_implementation(sten.GroupedNMSparsifier, torch.Tensor, sten.GroupedNMTensor)(
        sten.GroupedNMSparsifier(2, 4, 16, sparse_dim=1, group_dim=0), whole((R, T), torch.float16, 1).to(DEV).requires_grad_(True))
    B, go = whole((T, C), torch.float16, 2).to(DEV), whole((R, C), torch.float16, 3)
    torch.mm(w, B).backward(go.to(DEV))
    assert within(w.grad.wrapped_tensor.to_dense(), to_np(go).astype(np.float64) @ to_np(B).astype(np.float64).T, 0.0, torch.float16)
