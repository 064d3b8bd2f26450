"""Products with both dense operands transposed (torch.mm on B as it lies) on every tile, against float64."""
import pytest
import torch

import sten_amd as sten

DEV = "cuda:0"
# one rounding of the result, fp32 sums
BOUND = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


# 128 x 128, 256 x 128 and 256 x 256 tiles (by the rules of smfmac_tile and dense16_tile), each with extents that end inside one; reductions
# of 1 step to two turns of the ring of loads and a step more
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,N", [(128, 128), (200, 136), (1000, 24), (4096, 2048), (4000, 2040), (4104, 4104)])
@pytest.mark.parametrize("C", [64, 320, 704])
def test_torch_mm_as_it_lies(R, C, N, dtype):
    print(f"case tt tiles {dtype} R={R} C={C} N={N}", flush=True)
    g = torch.Generator(DEV).manual_seed(R + C + N)
    W = (torch.randn(R, C, device=DEV, generator=g) * 0.1).to(dtype)
    w = sten.GroupedNMTensor.from_dense(W, 2, 4, sparse_dim=1, group_size=16, group_dim=0)
    Wd = w.to_dense().double()
    B = torch.randn(C, N + 8, device=DEV, generator=g).to(dtype)[:, :N]      # (a pitch of its own)
    ref = Wd @ B.double()
    for name, c in (("sparse cores", sten.spmm_tt(w, B)), ("dense cores", sten.spmm_tt_dense(w, B, reduce_dim=1))):
        assert c.shape == (R, N)
        assert ((c.double() - ref).norm() / ref.norm()).item() <= BOUND[dtype], name
    Gy = torch.randn(R, N, device=DEV, generator=g).to(dtype)
    gb = sten.spmm_tt_dense(w, Gy, reduce_dim=0)
    ref = Wd.t() @ Gy.double()
    assert ((gb.double() - ref).norm() / ref.norm()).item() <= BOUND[dtype]
