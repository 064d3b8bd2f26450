"""Products with both dense operands transposed (torch.mm on B as it lies) on every tile, against float64."""
import pytest
import torch
from torch.profiler import ProfilerActivity, profile

import sten_amd as sten

DEV = "cuda:0"
# one rounding of the result, fp32 sums
BOUND = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def check(c, a, b, dtype, name):
    """Every element: the rounding of the result (half of the smallest subnormal where it is below the normal numbers) and the fp32 sum's, of K
    products in any order at most K 2^-24 times the sum of their magnitudes (twice that: the matrix cores may cut instead of round)."""
    ref = a.double() @ b.double()
    assert c.shape == ref.shape
    assert ((c.double() - ref).norm() / ref.norm()).item() <= BOUND[dtype], name
    bound = BOUND[dtype] * ref.abs() + 2.0 ** -23 * b.shape[0] * (a.double().abs() @ b.double().abs()) + 2.0 ** -25
    off = (c.double() - ref).abs() > bound      # (a NaN is not, but the norm above has seen it)
    assert not bool(off.any()), f"{name}: {int(off.sum())} elements, the first at {off.nonzero()[0].tolist()}"


def operands(R, C, N, dtype):
    g = torch.Generator(DEV).manual_seed(R + C + N)
    W = (torch.randn(R, C, device=DEV, generator=g) * 0.1).to(dtype)
    w = sten.GroupedNMTensor.from_dense(W, 2, 4, sparse_dim=1, group_size=16, group_dim=0)
    # (a pitch of its own, and no numbers behind the rows: what is read there must not show)
    wide = torch.full((C, (N + 7) // 8 * 8 + 8), float("nan"), device=DEV, dtype=dtype)
    B = wide[:, :N]
    B.copy_(torch.randn(C, N, device=DEV, generator=g))
    return w, B, g


# Tiles of 128 x 128 and 256 x 128, of 256 x 256 on the sparse cores (2240 rows) and on both (2240 rows and as many of B), each with extents that end
# inside one; reductions of 1 step to two turns of the ring of loads and some steps more (64 positions a step; a turn is 7 steps on 128 x 128 tiles, else 4)
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,N,C", [(R, N, C) for R, N in [(128, 128), (200, 136), (1000, 24), (4096, 2048), (4000, 2040), (4104, 4104)] for C in (64, 320, 704)]
                         + [(200, 136, 1088), (1000, 30, 1088), (2240, 3880, 64), (2240, 3880, 320), (2240, 3877, 704), (2240, 3880, 2240)])
def test_torch_mm_as_it_lies(R, C, N, dtype):
    print(f"case tt tiles {dtype} R={R} C={C} N={N}", flush=True)
    w, B, g = operands(R, C, N, dtype)
    Wd = w.to_dense()
    check(sten.spmm_tt(w, B), Wd, B, dtype, "sparse cores")
    check(sten.spmm_tt_dense(w, B, reduce_dim=1), Wd, B, dtype, "dense cores")
    Gy = torch.randn(R, N, device=DEV, generator=g).to(dtype)
    check(sten.spmm_tt_dense(w, Gy, reduce_dim=0), Wd.t(), Gy, dtype, "dense cores, transposed weight")


# A last row that ends with the storage, inside a piece of 8 columns, is not read as it lies.
@pytest.mark.gpu
@pytest.mark.parametrize("N", [17, 30, 133])
def test_storage_that_ends_with_the_last_row(N):
    w, B, _ = operands(256, 128, N, torch.float16)
    pitch = B.stride(0)
    short = torch.empty(127 * pitch + N, device=DEV, dtype=torch.float16).as_strided((128, N), (pitch, 1))
    short.copy_(B)
    print(f"case tt short storage N={N}", flush=True)
    sten.spmm_tt(w, short), sten.spmm_tt_dense(w, short, reduce_dim=1)      # (packs the operands)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        c, d = sten.spmm_tt(w, short), sten.spmm_tt_dense(w, short, reduce_dim=1)
        torch.cuda.synchronize()
    check(c, w.to_dense(), B, torch.float16, "sparse cores")
    check(d, w.to_dense(), B, torch.float16, "dense cores")
    names = [e.name for e in p.events() if "nmg::" in e.name]
    if names:      # a copy and a product each
        assert len(names) == 4, names


# Which tiles those extents take: outputs and columns as (sparse, dense) kernels name them.
@pytest.mark.gpu
@pytest.mark.parametrize("R,N,C,sparse,dense", [
    (200, 136, 1088, "1, 4, 4, 1, 1", "8, 2, true, true, false, 2"),           # 128 x 128
    (4104, 4104, 704, "2, 4, 4, 1, 2", "8, 2, true, true, false, 4"),          # 256 x 128
    (2240, 3880, 320, "2, 8, 4, 1, 4", "8, 2, true, true, false, 4"),          # 256 x 256 / 256 x 128
    (2240, 3880, 2240, "2, 8, 4, 1, 4", "16, 4, true, true, false, 4"),        # 256 x 256
])
def test_tiles_that_the_products_take(R, N, C, sparse, dense):
    print(f"case tt tiles taken R={R} C={C} N={N}", flush=True)
    w, B, _ = operands(R, C, N, torch.float16)
    for kernel, sizes, call in (("spmm_smfmac_direct_kernel", sparse, lambda: sten.spmm_tt(w, B)),
                                ("dense16_direct_kernel", dense, lambda: sten.spmm_tt_dense(w, B, reduce_dim=1))):
        call()
        torch.cuda.synchronize()
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            call()
            torch.cuda.synchronize()
        names = [e.name for e in p.events() if "nmg::" in e.name]
        if not names:
            pytest.skip("the profiler reports no kernels")
        assert any(f"{kernel}<__half, {sizes}, " in name for name in names), names
