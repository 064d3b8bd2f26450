"""The direct kernels where the XCDs start their walk of the reduction apart (one round of workgroups, 64 K steps and more)."""
import numpy as np
import pytest
import torch

import sten_amd as sten
from helpers import rel_l2, seeded, to_np

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C,T,n,m,g,sd,rd,slices", [
    (512, 4096, 130, 2, 4, 16, 1, 1, 1),      # 64 steps: the fewest that start apart; sparse cores
    (512, 4224, 130, 2, 4, 16, 1, 1, 1),      # 66 steps: no multiple of the eight starts or of the four stages
    (300, 4032, 130, 2, 4, 16, 1, 1, 1),      # 63 steps: all from the first
    (256, 8384, 40, 2, 4, 16, 1, 1, 2),       # slices of 66 and 65 steps: the starts follow each slice
    (4096, 512, 130, 2, 4, 16, 1, 0, 1),      # dense cores, reduction along the group dim
    (512, 4224, 130, 4, 8, 4, 1, 1, 1),       # dense cores, reduction along the sparse dim
    (8384, 256, 40, 2, 4, 16, 1, 0, 2),
    (4224, 33, 300, 2, 8, 4, 0, 0, 1),
])
def test_every_step_of_the_reduction_once(dtype, R, C, T, n, m, g, sd, rd, slices):
    print(f"case {dtype} {R}x{C} T={T} {n}:{m}:{g} sparse_dim={sd} reduce_dim={rd} slices={slices}", flush=True)
    # whole numbers up to 3: every partial sum of up to 8384 products is below 2^24, so single precision is exact
    # in any order and only the rounding of the result is left: 2^-11 of a value in fp16, 2^-8 in bf16
    W = torch.randint(-3, 4, (R, C), generator=torch.Generator().manual_seed(R + C + T)).to(dtype)
    x = torch.randint(-3, 4, (T, C if rd == 1 else R), generator=torch.Generator().manual_seed(1)).to(dtype)
    w = sten.GroupedNMTensor.from_dense(W.to(DEV), n, m, sparse_dim=sd, group_size=g, group_dim=1 - sd)
    w.spmm_opt["slices"] = slices
    D = to_np(w.to_dense()).astype(np.float64)
    ref = to_np(x).astype(np.float64) @ (D.T if rd == 1 else D)
    y = to_np(sten.spmm(w, x.to(DEV), reduce_dim=rd)).astype(np.float64)
    bound = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * np.abs(ref)
    assert (np.abs(y - ref) <= bound).all()


@pytest.mark.parametrize("sd", [0, 1])
def test_matrix_product_and_its_gradients(sd):
    # torch.mm with 66 K steps in one of its products: transposed copies, the dense product of row operands
    for R, C, N in ((512, 4224, 264), (4224, 512, 264), (512, 512, 4224)):
        W = seeded((R, C), torch.float16, seed=R, std=0.02)
        w = sten.get_sparsifier_implementation(sten.GroupedNMSparsifier, torch.Tensor, sten.GroupedNMTensor)(
            sten.GroupedNMSparsifier(2, 4, 16, sparse_dim=sd, group_dim=1 - sd), W.to(DEV).requires_grad_(True))
        D = w.wrapped_tensor.to_dense().double()
        B = seeded((C, N), torch.float16, seed=2).to(DEV).requires_grad_(True)
        go = seeded((R, N), torch.float16, seed=3).to(DEV)
        y = torch.mm(w, B)
        y.backward(go)
        assert rel_l2(to_np(y), to_np(D @ B.detach().double())) <= 1e-3
        assert rel_l2(to_np(B.grad), to_np(D.t() @ go.double())) <= 1e-3
        assert rel_l2(to_np(w.grad.wrapped_tensor.to_dense()), to_np(go.double() @ B.detach().double().t())) <= 1e-3


def bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C,T,n,m,g,rd,opt", [
    (4096, 4224, 2000, 2, 4, 16, 1, {}),                   # 256 x 128 on the sparse cores, several bands of tiles
    (4096, 4224, 777, 2, 4, 16, 1, {}),
    (512, 4224, 2100, 2, 4, 16, 1, {"slices": 1}),         # one band
    (1100, 8448, 300, 2, 4, 16, 1, {"slices": 2}),
    (2048, 4224, 2000, 4, 8, 4, 1, {}),                    # dense cores
    (1100, 4224, 500, 4, 8, 4, 1, {"slices": 1}),
    (4224, 2048, 600, 2, 4, 16, 0, {"slices": 1}),
    (8448, 1100, 300, 2, 4, 16, 0, {"slices": 2}),
])
def test_a_row_of_activations_gives_the_same_bits_in_every_tile(R, C, T, n, m, g, rd, opt, dtype):
    print(f"case {dtype} {R}x{C} T={T} {n}:{m}:{g} reduce_dim={rd} {opt}", flush=True)
    w = sten.GroupedNMTensor.from_dense(seeded((R, C), dtype, seed=1).to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
    w.spmm_opt.update(opt)
    x = seeded((1, C if rd == 1 else R), dtype, seed=2).to(DEV).expand(T, -1).contiguous()
    y = bits(sten.spmm(w, x, reduce_dim=rd))
    assert bool((y == y[:1]).all())
    if rd == 1:
        c = bits(sten.spmm_tt(w, x.t().contiguous()))
        assert bool((c == c[:, :1]).all())


@pytest.mark.parametrize("n,m,g,name,variants", [(2, 4, 16, "variant", (6, 8)), (4, 8, 4, "dense_variant", (0, 1))])
def test_tiles_asked_for_by_number_keep_the_order_of_the_reduction(n, m, g, name, variants):
    w = sten.GroupedNMTensor.from_dense(seeded((1100, 4224), torch.float16, seed=1).to(DEV), n, m, sparse_dim=1, group_size=g, group_dim=0)
    x, got = seeded((600, 4224), torch.float16, seed=2).to(DEV), []
    for v in variants:
        w.spmm_opt[name] = v
        got.append(bits(sten.spmm(w, x, reduce_dim=1)))
    assert torch.equal(*got)
